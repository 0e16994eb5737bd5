/* SPDX-License-Identifier: Apache-2.0 */
/**
 * @file   silu_ref.h
 * @brief  The expert activation's sigmoid, for the device and for the host program that compares it with the
 *         library's double functions over every float (tests/test_silu.py).
 */
#ifndef HIPQ_SILU_REF_H
#define HIPQ_SILU_REF_H

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define HIPQ_SILU_FN __device__ __forceinline__
#else
#define HIPQ_SILU_FN static inline
#endif

/* sigmoid(g) * g with the sigmoid in double on the float-rounded exponential, as the reference:
 *   en = float(exp(double(-g))), sig = float(1.0 / (1.0 + double(en))).
 * Both double results are only kept to float, so neither needs the library's last-bit exp and
 * division (about a hundred double instructions a value; in the products of many tokens they were
 * half of a workgroup's time outside its loop). exp: 2^k e^r with r = x - k ln 2 in two fused steps,
 * |r| < 0.3466, and e^r = 1 + r + r^2 q(r) with q of degree 9 through the ten Chebyshev nodes of that range (its
 * first coefficient a half, a constant of the instruction set), in two chains. That is off by 2^-54.6 at most; the
 * Taylor sum to r^11 is off by 2^-47, and two of all floats had another exponential. Division: a reciprocal of 22 bits
 * or better and one cubic step y (1 + e + e^2), e = 1 - d y.
 * Both round to the library forms' float for every float from 2^-30 to 250 in magnitude, with glibc's exp as the
 * library form. Beyond +-200 the exponential is 0 or infinite as a float. */
template <typename Rcp> HIPQ_SILU_FN float hipq_silu_ref(float g, Rcp rcp) {
  const double x = (double)fminf(fmaxf(-g, -200.f), 200.f);
  const double kbig = fma(x, 1.4426950408889634, 6755399441055744.0); /* 1.5 * 2^52: k in the low bits */
  const double k = kbig - 6755399441055744.0;
  const double r = fma(k, -2.3190468138462996e-17, fma(k, -0.6931471805599453, x));
  const double r2 = r * r;
  double even = 0x1.28917e2c43a66p-22, odd = 0x1.af38a0d2d9620p-26; /* coefficients of r^10, r^11 and down */
  constexpr double E[4] = {0x1.a019b9133a48ap-16, 0x1.6c16c1788a49bp-10, 0x1.5555555553d67p-5, 0.5};
  constexpr double O[4] = {0x1.71de0db21e27fp-19, 0x1.a01a01a7c327ap-13, 0x1.11111111109b4p-7, 0x1.5555555555556p-3};
#pragma unroll
  for (int i = 0; i < 4; ++i) even = fma(even, r2, E[i]), odd = fma(odd, r2, O[i]);
  const double p = 1.0 + fma(r2, fma(odd, r, even), r);
  const uint64_t bits = __builtin_bit_cast(uint64_t, p) + (__builtin_bit_cast(uint64_t, kbig) << 52);
  const float en = (float)__builtin_bit_cast(double, bits);
  const double d = 1.0 + (double)en;
  const double y = rcp(d);
  const double e = fma(-d, y, 1.0);
  const float sig = en == INFINITY ? 0.f : (float)fma(y, fma(e, e, e), y);
  return sig * g;
}

#endif /* HIPQ_SILU_REF_H */
