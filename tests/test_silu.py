"""CPU: the polynomial and the reciprocal step of the expert activation (csrc/silu_ref.h) give the reference's float,
sigmoid(g) * g with exp and the division in double, for every float."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "silu_ref.h"
#include <cstdio>
#include <cstring>
#include <initializer_list>
static uint32_t bits(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static float value(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static float library(float g) { /* the reference: sigmoid in double on the rounded exponential */
  const float en = (float)exp(-(double)g);
  return (float)(1.0 / (1.0 + (double)en)) * g;
}
static bool same(float a, float b) { return bits(a) == bits(b) || (a != a && b != b); }
int main() {
  long wrong = 0, seen = 0;
  const uint32_t lo = bits(0x1p-30f), hi = bits(250.f);
#pragma omp parallel for reduction(+ : wrong, seen) schedule(static, 1 << 16)
  for (uint32_t i = lo; i <= hi; ++i)
    for (uint32_t s = 0; s < 2; ++s) {
      const float g = value(i | s << 31), want = library(g);
      /* the hardware's reciprocal has 24 bits; three of 22, off to either side */
      for (double off : {1.0, 1.0 + 0x1p-22, 1.0 - 0x1p-22})
        wrong += !same(hipq_silu_ref(g, [=](double d) { return (double)(1.0f / (float)d) * off; }), want);
      ++seen;
    }
  for (float g : {0.f, -0.f, 1e-30f, -1e-30f, 1e-45f, 251.f, -251.f, 1e30f, -1e30f, INFINITY, -INFINITY, NAN})
    wrong += !same(hipq_silu_ref(g, [](double d) { return (double)(1.0f / (float)d); }), library(g)), ++seen;
  printf("%ld %ld\n", wrong, seen);
}
"""


def test_silu_series_rounds_to_the_library_forms_float(tmp_path):
    src = tmp_path / "silu.cpp"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-mavx2", "-mfma", "-ffp-contract=off", "-fopenmp", "-I",
                    os.path.join(ROOT, "nntrainer_amd", "csrc"), str(src), "-o", str(tmp_path / "silu")], check=True)
    out = subprocess.run([str(tmp_path / "silu")], capture_output=True, text=True, check=True, timeout=600).stdout.split()
    assert int(out[1]) > 600e6 and int(out[0]) == 0, "%s of %s floats differ" % tuple(out)
