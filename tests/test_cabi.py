"""CPU: the C-ABI library loads, exports every symbol include/hipq.h declares, and
fails loudly (no fallback) where there is no GPU."""
import functools
import os
import re
import sys

import pytest

from nntrainer_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "hipq.h")).read()
    return sorted(set(re.findall(r"HIPQ_API\s+[\w\s\*]+?\b(hipq_\w+)\s*\(", text)))


def test_header_symbols_are_exported():
    names = _declared()
    assert len(names) >= 15 and set(names) == set(capi.SYMBOLS)
    lib = capi.lib()
    for n in names:
        assert getattr(lib, n) is not None


def test_product_library_exports_exactly_the_header(tmp_path):
    """libhipq.so exports the functions include/hipq.h declares and no others; the measurement
    and test helpers live in libhipq_bench.so, which links it."""
    import subprocess
    out = subprocess.run(["nm", "-D", "--defined-only", capi.LIB_PATH], capture_output=True, text=True, check=True).stdout
    exported = sorted(line.split()[-1] for line in out.splitlines() if " T " in line)
    assert exported == _declared(), set(exported) ^ set(_declared())
    bench = os.path.join(os.path.dirname(capi.LIB_PATH), "libhipq_bench.so")
    out = subprocess.run(["nm", "-D", "--defined-only", bench], capture_output=True, text=True, check=True).stdout
    have = {line.split()[-1] for line in out.splitlines() if " T " in line}
    assert set(capi.BENCH_SYMBOLS) <= have
    needed = subprocess.run(["readelf", "-d", bench], capture_output=True, text=True, check=True).stdout
    assert "libhipq.so" in needed


def test_weight_size_rules():
    # 18 B / 32, 144 B / 256, 210 B / 256 (q4_0_tensor.h:20-31, q4_k_tensor.h:25-33, q6_k_tensor.h:25-32)
    assert capi.weight_nbytes("q4_0", 4096, 4096) == 9437184
    assert capi.weight_nbytes("q4_K", 12288, 4096) == 28311552
    assert capi.weight_nbytes("q6_K", 151936, 4096) == 510504960
    for kind, k in (("q4_0", 48), ("q4_K", 128), ("q6_K", 300)):
        with pytest.raises(capi.HipqError) as e:
            capi.weight_nbytes(kind, 8, k)
        assert e.value.code == -1


def test_model_file_offsets_follow_the_reference_rule():
    """MODEL_FORMAT_BIN is the graph's tensors back to back; only tensors with
    quantization parameters other than Q4_0 / Q6_K carry a 16-bit scheme word in front
    (models/neuralnet.cpp:696-703). Host arithmetic: no device needed."""
    tensors = [("skip", 151936 * 1024 * 4),            # fp32 embedding
               ("skip", 1024 * 4),                     # a norm's gamma
               ("q4_0", 2048, 1024, capi.LAYOUT_X8),
               ("q4_K", 3072, 1024, capi.LAYOUT_X8),
               ("q4_K", 1024, 3072, capi.LAYOUT_X8),
               ("q6_K", 151936, 1024)]
    offs, end = capi.file_layout(tensors, offset=16)
    want, at = [], 16
    for t in tensors:
        if t[0] == "skip":
            want.append(at)
            at += t[1]
            continue
        if t[0] == "q4_K":
            at += 2
        want.append(at)
        at += capi.weight_nbytes(t[0], t[1], t[2])
    assert offs == want and end == at
    assert capi.file_layout([], offset=5) == ([], 5)
    with pytest.raises(capi.HipqError):
        capi.file_layout([("q4_K", 8, 100)])
    with pytest.raises(capi.HipqError):
        capi.file_layout([("skip", -1)])


def test_no_gpu_means_loud_failure():
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    with pytest.raises(capi.HipqError):
        capi.init(0)
    import numpy as np
    blocks = np.zeros(capi.weight_nbytes("q4_0", 8, 32), np.uint8)
    with pytest.raises(capi.HipqError) as e:
        capi.Weight("q4_0", 8, 32, blocks)
    assert e.value.code == -2  # HIPQ_ERR_NOT_INITIALIZED: nothing computes without the device
    with pytest.raises(capi.HipqError) as e:
        capi.weights_from_file("/nonexistent", [("q4_0", 8, 32)])
    assert e.value.code == -2


@pytest.mark.parametrize("name,args,kwargs,error", [
    ("matmul", (None, 1), {}, TypeError),                              # 'm' and 'c' missing
    ("matmul", (None, 1, 1, 1), {"rows": 1}, TypeError),               # no such keyword
    ("matmul", (None, 1, 1, 1), {"m": 1}, TypeError),                  # given twice
    ("matmul", (None,) + (1,) * 8, {}, TypeError),                     # too many
    ("matmul", (None, 1, 1, 1), {}, AttributeError),                   # not a weight
    ("matmul_multi", ([], 1, 1, []), {}, ValueError),                  # no weights
    ("matmul_multi", (None, 1, 1, None), {}, TypeError),               # not sequences
    ("mlp_swiglu_down", (None, None, None, 1, 1), {}, TypeError),      # 'out' missing
])
def test_native_calls_check_their_arguments(name, args, kwargs, error):
    capi.lib()
    with pytest.raises(error):
        getattr(capi, name)(*args, **kwargs)


class _Calls:
    """The matmul calls bound to a stub that notes what each entry point is given."""

    def __enter__(self):
        import ctypes as C
        self.lib = capi.lib()
        self.args, one = None, [C.c_void_p, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_int64]
        kinds = {"matmul": one + [C.c_int, C.c_void_p], "matmul_each_row": one + [C.c_int, C.c_void_p], "matmul_noalloc": one + [C.c_void_p],
                 "matmul_multi": [C.c_int, C.c_void_p, C.c_void_p, C.c_int64, C.c_int64, C.c_void_p, C.c_void_p, C.c_int, C.c_void_p],
                 "mlp_swiglu": [C.c_void_p] + one + [C.c_int, C.c_void_p], "mlp_swiglu_down": [C.c_void_p] * 2 + one + [C.c_int, C.c_void_p]}

        def note(name, *args):
            self.args = [a or 0 for a in args]
            if name == "matmul_multi":  # arrays of handles, outputs and strides
                for i, t in ((1, C.c_void_p), (5, C.c_void_p), (6, C.c_int64)):
                    self.args[i] = list((t * args[0]).from_address(args[i]))
            return 0

        class Stub:
            pass
        for name, types in kinds.items():
            f = C.CFUNCTYPE(C.c_int, *types)(functools.partial(note, name))
            setattr(Stub, "hipq_" + name, f)
        capi._lib = Stub
        capi._bind_native(Stub)
        return self

    def __exit__(self, *exc):
        capi._lib = self.lib
        capi._bind_native(self.lib)


class _Shape:  # a weight's fields
    n, k = 8, 32

    def __init__(self, address):
        import ctypes as C
        self.handle = C.c_void_p(address)


class _Stream:
    def __init__(self, parameter):
        self._as_parameter_ = parameter


def test_native_calls_take_the_streams_ctypes_takes():
    import ctypes as C
    import numpy as np
    forms = [(None, 0), (0, 0), (0x30, 0x30), (C.c_void_p(0x30), 0x30), (C.c_void_p(None), 0), (_Stream(C.c_void_p(0x40)), 0x40),
             (_Stream(0x50), 0x50)]
    w = _Shape(16)
    with _Calls() as calls:
        for stream, want in forms:
            for name, args in (("matmul", (w, 64, 2, 128)), ("matmul_each_row", (w, 64, 2, 128)), ("matmul_noalloc", (w, 64, 2, 128)),
                               ("matmul_multi", ([w], 64, 2, [128])), ("mlp_swiglu", (w, w, 64, 2, 128)),
                               ("mlp_swiglu_down", (w, w, w, 64, 2, 128))):
                getattr(capi, name)(*args, stream=stream)
                assert calls.args[-1] == want, (name, stream)
        for stream in (np.int64(0x30), np.zeros(4), object(), 1.5):
            calls.args = None
            with pytest.raises((TypeError, C.ArgumentError)):
                capi.matmul(w, 64, 2, 128, stream=stream)
            assert calls.args is None


def test_native_calls_take_the_buffers_the_binding_takes():
    import ctypes as C
    import numpy as np
    import torch
    w, a = _Shape(16), np.zeros((4, 64), np.float32)
    w._h = w.handle  # capi.Weight's own field
    read_only = np.zeros(64, np.float32)
    read_only.flags.writeable = False
    t = torch.zeros(64)
    forms = [(None, 0), (64, 64), (a, a.ctypes.data), (a[1:, 3:], a.ctypes.data + 4 * 67), (a[:, ::2], a.ctypes.data),
             (read_only, read_only.ctypes.data), (t[5:], t.data_ptr() + 20), (a.view(np.recarray), a.ctypes.data)]
    with _Calls() as calls:
        for x, want in forms:
            capi.matmul(w, x, 2, x)
            assert calls.args == [16, want, 2, 32, want, 8, capi.MEM_DEVICE, 0]
        capi.matmul(w, 64, C.c_int64(2), 128, lda=C.c_int64(48), ldc=np.int64(16), mem=C.c_int(0))
        assert calls.args == [16, 64, 2, 48, 128, 16, 0, 0]
        for x in (np.int64(64), np.float32(1), b"0123456789abcdef", bytearray(16), memoryview(b"01234567"), C.c_void_p(64),
                  (C.c_float * 4)(), object()):
            for args in ((w, x, 2, 128), (w, 64, 2, x)):
                calls.args = None
                with pytest.raises(AttributeError):
                    capi.matmul(*args)
                assert calls.args is None, x


def test_ctypes_forms_make_the_same_calls():
    """An interpreter without the native module uses the ctypes forms: the same entry points, arguments and defaults."""
    import numpy as np
    w, x, y = _Shape(16), _Shape(24), np.zeros((2, 32), np.float32)
    y_at = y.ctypes.data
    cases = [("matmul", (w, y, 2, 128), {}), ("matmul", (w, y, 2, 128, 40), {"ldc": 0, "mem": 0, "stream": 0x30}),
             ("matmul_each_row", (w, 64, 2, y), {"lda": None, "ldc": 16}), ("matmul_noalloc", (w, 64), {"m": 1, "c": y, "stream": None}),
             ("matmul_multi", ([w, x], y, 3, (y, 128)), {"lda": 64}), ("matmul_multi", ((w,), 64, 1, [y], [9], 0, 0x30), {}),
             ("mlp_swiglu", (w, x, y, 2, 128, 33), {"ldo": 10}), ("mlp_swiglu_down", (w, x, w, y, 2, 128), {"stream": 0x30})]
    with _Calls() as calls:
        for name, args, kwargs in cases:
            seen = []
            for form in (getattr(capi, name), capi._FORMS[name]):
                assert form(*args, **kwargs) is None
                seen.append(calls.args)
            assert seen[0] == seen[1], (name, seen)
            assert y_at in seen[0] or y_at in seen[0][5]


def test_native_module_is_built_per_interpreter_and_optional(tmp_path):
    import subprocess
    import sysconfig
    lib = os.path.dirname(capi.LIB_PATH)
    assert os.path.exists(os.path.join(lib, "hipq_native" + sysconfig.get_config_var("EXT_SUFFIX")))
    # no interpreter, no headers: the library's own targets remain
    out = subprocess.run(["make", "-B", "-n", "-C", capi.CSRC, "PYTHON=/nonexistent"], capture_output=True, text=True, check=True).stdout
    assert "libhipq.so" in out and "native_calls" not in out
    # without the module the binding loads and calls through ctypes
    code = ("import importlib.machinery as m; m.EXTENSION_SUFFIXES.insert(0, '.other-abi.so')\n"
            "import warnings; warnings.simplefilter('error')\n"
            "from nntrainer_amd import capi\n"
            "try: capi.lib()\n"
            "except RuntimeWarning: print(capi.matmul.__module__)\n")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT)
    assert r.stdout.split() == ["nntrainer_amd.capi"], r.stderr


def test_native_calls_follow_the_headers_signatures(tmp_path):
    import subprocess
    import sysconfig
    text = open(os.path.join(ROOT, "include", "hipq.h")).read()
    for n, (old, new) in enumerate([("", ""), (r"hipq_matmul\((hipq_weight_t w), ", r"hipq_matmul(\1, int flags, "),
                                    ("const int64_t \\*ldc", "const int32_t *ldc")]):
        changed = re.sub(old, new, text) if old else text
        assert not old or changed != text, old
        d = tmp_path / str(n)
        d.mkdir()
        (d / "hipq.h").write_text(changed)
        r = subprocess.run(["gcc", "-std=c11", "-fsyntax-only", "-Werror=incompatible-pointer-types", "-Werror=int-conversion", "-I", str(d),
                            "-I", sysconfig.get_paths()["include"], os.path.join(capi.CSRC, "native_calls.c")], capture_output=True, text=True)
        assert (r.returncode == 0) == (not old), (old, r.stderr)


def test_product_never_imports_the_oracle():
    """The package and the library sources must not reach into oracle/."""
    for base, _, files in os.walk(os.path.join(ROOT, "nntrainer_amd")):
        for f in files:
            if f.endswith((".py", ".hip", ".h", ".c", ".cpp", "Makefile")):
                text = open(os.path.join(base, f), errors="ignore").read()
                assert "oracle" not in text.lower().replace("oracle/_ref", ""), os.path.join(base, f)
