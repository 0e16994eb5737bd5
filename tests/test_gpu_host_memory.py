"""Host-memory operands of the C ABI (HIPQ_MEM_HOST): pageable memory goes through the library's
pinned staging ring, page-locked memory (hipq_host_alloc, what the context's MemAllocator hands
the framework, cl_context.cpp:83) by DMA as it is. Both must give the bits of the device-memory
call. Also: the multi-weight call on host memory, and releasing a stream's scratch."""
import ctypes

import numpy as np
import pytest

from nntrainer_amd import capi, synth

pytestmark = pytest.mark.gpu


def _device_result(w, a):
    import gpu_util as gu
    return gu.gpu_matmul(w, a)


@pytest.mark.parametrize("kind,m,k,n,lda_pad,ldc_pad", [
    ("q4_0", 700, 1024, 3000, 0, 0),     # A 2.8 MB, C 8.4 MB: several slices of the ring each way
    ("q4_0", 700, 1024, 3000, 32, 8),    # strided rows on both sides
    ("q4_K", 37, 2048, 1024, 0, 0),
    ("q6_K", 1, 1024, 5000, 0, 0),       # decode row
    ("q4_0", 1, 32, 600000, 0, 0),       # one output row longer than a ring slot (2.4 MB)
])
def test_pageable_operands_give_the_device_bits(hipq, cr, kind, m, k, n, lda_pad, ldc_pad):
    blocks = cr.quantize_weights(cr.oracle(), kind, synth.normal(9000 + n % 97, (n, k), 0.02))
    w = capi.Weight(kind, n, k, blocks)
    a = synth.normal(9001 + m, (m, k))
    want = _device_result(w, a)
    lda, ldc = k + lda_pad, n + ldc_pad
    a_host = np.full((m, lda), np.float32(7e9))
    a_host[:, :k] = a
    c_host = np.full((m, ldc), np.float32(-3.5))
    for _ in range(2):  # the second call finds ring slots and operand buffers in use before
        c_host[:, :n] = np.nan
        capi.matmul(w, a_host, m, c_host, lda=lda, ldc=ldc, mem=capi.MEM_HOST)
        assert np.array_equal(c_host[:, :n].view(np.uint32), want.view(np.uint32))
        assert np.all(c_host[:, n:] == np.float32(-3.5)), "the padding of the output rows was written"
    w.destroy()


def test_page_locked_operands(hipq, cr):
    kind, m, k, n = "q4_K", 64, 1024, 768
    blocks = cr.quantize_weights(cr.oracle(), kind, synth.normal(9100, (n, k), 0.02))
    w = capi.Weight(kind, n, k, blocks)
    a = synth.normal(9101, (m, k))
    want = _device_result(w, a)
    pa, pc = capi.host_alloc(m * k * 4), capi.host_alloc(m * n * 4)
    try:
        a_pin = np.ctypeslib.as_array(ctypes.cast(pa, ctypes.POINTER(ctypes.c_float)), (m, k))
        c_pin = np.ctypeslib.as_array(ctypes.cast(pc, ctypes.POINTER(ctypes.c_float)), (m, n))
        assert not a_pin.any() and not c_pin.any(), "the allocator hands out zero-filled memory"
        a_pin[:] = a
        capi.matmul(w, pa, m, pc, mem=capi.MEM_HOST)
        assert np.array_equal(c_pin.view(np.uint32), want.view(np.uint32))
    finally:
        capi.host_free(pa)
        capi.host_free(pc)
        capi.host_free(None)
    w.destroy()


@pytest.mark.parametrize("kind,m", [("q4_0", 1), ("q4_0", 19), ("q4_K", 1), ("q6_K", 3)])
def test_multi_weight_call_on_host_memory(hipq, cr, kind, m):
    """hipq_matmul_multi with host operands: the activation crosses once and the products run as
    for device memory; same bits as one hipq_matmul per weight."""
    k, ns = 1024, (512, 256, 384)
    ws = [capi.Weight(kind, n, k, cr.quantize_weights(cr.oracle(), kind, synth.normal(9200 + n, (n, k), 0.02)))
          for n in ns]
    a = synth.normal(9201 + m, (m, k))
    cs = [np.full((m, n), np.nan, np.float32) for n in ns]
    capi.matmul_multi(ws, a, m, cs, mem=capi.MEM_HOST)
    for w, c in zip(ws, cs):
        assert np.array_equal(c.view(np.uint32), _device_result(w, a).view(np.uint32))
        w.destroy()


def test_stream_release(hipq, cr):
    """A stream's scratch can be given back and comes again with the next call."""
    import gpu_util as gu
    import torch
    kind, m, k, n = "q4_K", 16, 1024, 512
    w = capi.Weight(kind, n, k, cr.quantize_weights(cr.oracle(), kind, synth.normal(9300, (n, k), 0.02)))
    a = synth.normal(9301, (m, k))
    want = _device_result(w, a)
    st = torch.cuda.Stream()
    da = gu.dev(a)
    torch.cuda.synchronize()
    for _ in range(2):
        dc = torch.full((m, n), float("nan"), device="cuda")
        torch.cuda.synchronize()
        capi.matmul(w, da, m, dc, stream=st.cuda_stream)
        st.synchronize()
        assert np.array_equal(dc.cpu().numpy().view(np.uint32), want.view(np.uint32))
        capi.stream_release(st.cuda_stream)
    capi.stream_release(st.cuda_stream)  # nothing kept: a no-op
    w.destroy()


class _Pinned:
    """A float32 array in page-locked memory of the context's allocator."""

    def __init__(self, shape, fill=None):
        self.n = int(np.prod(shape))
        self.addr = capi.host_alloc(self.n * 4)
        self.arr = np.ctypeslib.as_array(ctypes.cast(self.addr, ctypes.POINTER(ctypes.c_float)), tuple(shape))
        if fill is not None:
            self.arr[...] = fill

    def free(self):
        capi.host_free(self.addr)


@pytest.mark.parametrize("kind,m,k,n,lda_pad,ldc_pad", [
    ("q4_0", 1, 1024, 3072, 0, 0),      # one launch that quantizes the row itself
    ("q4_K", 1, 4096, 4096, 0, 0),
    ("q6_K", 1, 1024, 40000, 0, 0),     # two launches (vocabulary-sized)
    ("q4_K", 3, 2048, 1024, 8, 4),      # strided rows on both sides
    ("q4_0", 8, 1024, 3072, 0, 12),
    ("q4_K", 8, 4096, 12288, 0, 0),     # the few-rows matrix-core kernel
    ("q4_0", 9, 1024, 3072, 0, 0),
    ("q4_K", 64, 4096, 4096, 0, 8),     # a short prefill chunk: 1 MiB each way
    ("q6_K", 100, 1024, 2048, 4, 0),
    ("q4_0", 128, 1024, 3072, 0, 0),    # the most rows this path takes
    ("q4_0", 129, 1024, 3072, 0, 0),    # one row more: through the copy engines
    ("q4_0", 100, 1024, 8192, 0, 0),    # outputs beyond 2 MiB: through the copy engines
])
def test_a_few_page_locked_rows_take_no_copy(hipq, cr, kind, m, k, n, lda_pad, ldc_pad):
    """Up to 128 rows and 2 MiB a side in page-locked memory (a decode step or a short chunk through the
    Layer API): the rows are
    fetched by a kernel and the product kernels write the host tensor directly. Same bits as the
    device-memory call; the padding of strided rows stays untouched; two calls in a row."""
    blocks = cr.quantize_weights(cr.oracle(), kind, synth.normal(9400 + n % 89, (n, k), 0.02))
    w = capi.Weight(kind, n, k, blocks)
    a = synth.normal(9401 + m, (m, k))
    want = _device_result(w, a)
    lda, ldc = k + lda_pad, n + ldc_pad
    pa, pc = _Pinned((m, lda), 7e9), _Pinned((m, ldc), -3.5)
    try:
        pa.arr[:, :k] = a
        for _ in range(2):
            pc.arr[:, :n] = np.nan
            capi.matmul(w, pa.addr, m, pc.addr, lda=lda, ldc=ldc, mem=capi.MEM_HOST)
            assert np.array_equal(pc.arr[:, :n].view(np.uint32), want.view(np.uint32))
            assert np.all(pc.arr[:, n:] == np.float32(-3.5))
        # the rows of a decode step of a batch: each with the bits of its own one-row product
        pc.arr[:, :n] = np.nan
        capi.matmul_each_row(w, pa.addr, m, pc.addr, lda=lda, ldc=ldc, mem=capi.MEM_HOST)
        for r in range(m):
            assert np.array_equal(pc.arr[r, :n].view(np.uint32), _device_result(w, a[r:r + 1])[0].view(np.uint32)), r
    finally:
        pa.free()
        pc.free()
        w.destroy()


@pytest.mark.parametrize("kind,m", [("q4_0", 1), ("q4_K", 1), ("q4_0", 4), ("q4_K", 8), ("q6_K", 2)])
def test_grouped_calls_on_a_few_page_locked_rows(hipq, cr, kind, m):
    """hipq_matmul_multi (Q, K, V) and hipq_mlp_swiglu (up, gate and the activation) with a decode
    step's page-locked operands: outputs written by the kernels, the bits of the device calls."""
    import gpu_util as gu
    import torch
    k, ns = 1024, (2048, 1024, 1024)
    ws = [capi.Weight(kind, n, k, cr.quantize_weights(cr.oracle(), kind, synth.normal(9500 + j, (n, k), 0.05)))
          for j, n in enumerate(ns)]
    a = synth.normal(9510 + m, (m, k))
    pa = _Pinned((m, k), a)
    pcs = [_Pinned((m, n), np.nan) for n in ns]
    po = _Pinned((m, ns[1]), np.nan)
    try:
        capi.matmul_multi(ws, pa.addr, m, [p.addr for p in pcs], mem=capi.MEM_HOST)
        dev = [torch.full((m, n), float("nan"), device="cuda") for n in ns]
        capi.matmul_multi(ws, gu.dev(a), m, dev, stream=gu.stream())
        torch.cuda.synchronize()
        for p, d in zip(pcs, dev):
            assert np.array_equal(p.arr.view(np.uint32), d.cpu().numpy().view(np.uint32))
        capi.mlp_swiglu(ws[1], ws[2], pa.addr, m, po.addr, mem=capi.MEM_HOST)
        want = torch.full((m, ns[1]), float("nan"), device="cuda")
        capi.mlp_swiglu(ws[1], ws[2], gu.dev(a), m, want, stream=gu.stream())
        torch.cuda.synchronize()
        assert np.array_equal(po.arr.view(np.uint32), want.cpu().numpy().view(np.uint32))
        # the whole MLP in one call: the hidden rows stay on the device, the output is written in place
        capi.mlp_swiglu_down(ws[1], ws[2], ws[0], pa.addr, m, pcs[0].addr, mem=capi.MEM_HOST)
        whole = torch.full((m, ns[0]), float("nan"), device="cuda")
        capi.matmul(ws[0], want, m, whole, stream=gu.stream())
        torch.cuda.synchronize()
        assert np.array_equal(pcs[0].arr.view(np.uint32), whole.cpu().numpy().view(np.uint32))
    finally:
        for p in [pa, po] + pcs:
            p.free()
        for w in ws:
            w.destroy()


@pytest.mark.parametrize("kind,m,k,n,pad", [
    ("q4_0", 1400, 1024, 3072, 0),      # five steps of 256 rows, the last of 376
    ("q4_0", 2100, 1024, 2048, 8),      # eight steps; strided rows on both sides
    ("q4_K", 700, 2048, 12288, 0),      # every step takes the prefill GEMM on whole K: two steps
    ("q4_K", 1100, 2048, 4096, 0),      # a step alone would be formed in parts of K, the whole call is not
    ("q6_K", 1100, 1024, 4096, 4),
    ("q6_K", 520, 3072, 8448, 0),       # likewise
    ("q4_0", 512, 1024, 3072, 0),       # outputs of 6 MB: one piece
])
def test_prefill_rows_in_steps_give_the_device_bits(hipq, cr, kind, m, k, n, pad):
    """512 rows and more in page-locked memory with outputs of 16 MiB and at least twice the input cross in
    steps of 256: a step's rows come in and the step before goes out while the kernels work. Every entry point that takes host rows gives the bits of its
    device-memory call on the whole matrix, twice in a row."""
    import gpu_util as gu
    import torch
    nd = 1024
    mk = lambda j, rows, cols: capi.Weight(kind, rows, cols, cr.quantize_weights(
        cr.oracle(), kind, synth.normal(9700 + j, (rows, cols), 0.05)))
    w, w2, wd = mk(0, n, k), mk(1, n, k), mk(2, nd, n)
    a = synth.normal(9710 + m, (m, k))
    lda, ldc = k + pad, n + pad
    pa = _Pinned((m, lda), 7e9)
    pa.arr[:, :k] = a
    pc, pc2, po, pd = _Pinned((m, ldc)), _Pinned((m, n)), _Pinned((m, n)), _Pinned((m, nd))
    try:
        da = gu.dev(a)
        want = torch.empty((m, n), device="cuda")
        want2 = torch.empty((m, n), device="cuda")
        capi.matmul_multi([w, w2], da, m, [want, want2], stream=gu.stream())
        single = torch.empty((m, n), device="cuda")
        capi.matmul(w, da, m, single, stream=gu.stream())
        act = torch.empty((m, n), device="cuda")
        capi.mlp_swiglu(w, w2, da, m, act, stream=gu.stream())
        down = torch.empty((m, nd), device="cuda")
        capi.mlp_swiglu_down(w, w2, wd, da, m, down, stream=gu.stream())
        torch.cuda.synchronize()
        bits = lambda t: t.cpu().numpy().view(np.uint32)
        for _ in range(2):
            pc.arr[...] = -3.5
            pc.arr[:, :n] = np.nan
            capi.matmul(w, pa.addr, m, pc.addr, lda=lda, ldc=ldc, mem=capi.MEM_HOST)
            assert np.array_equal(pc.arr[:, :n].view(np.uint32), bits(single))
            assert np.all(pc.arr[:, n:] == np.float32(-3.5)), "the padding of the output rows was written"
            pc.arr[...] = np.nan
            pc2.arr[...] = np.nan
            capi.matmul_multi([w, w2], pa.addr, m, [pc.addr, pc2.addr], lda=lda, ldc=[ldc, n], mem=capi.MEM_HOST)
            assert np.array_equal(pc.arr[:, :n].view(np.uint32), bits(want))
            assert np.array_equal(pc2.arr.view(np.uint32), bits(want2))
            po.arr[...] = np.nan
            capi.mlp_swiglu(w, w2, pa.addr, m, po.addr, lda=lda, mem=capi.MEM_HOST)
            assert np.array_equal(po.arr.view(np.uint32), bits(act))
            pd.arr[...] = np.nan
            capi.mlp_swiglu_down(w, w2, wd, pa.addr, m, pd.addr, lda=lda, mem=capi.MEM_HOST)
            assert np.array_equal(pd.arr.view(np.uint32), bits(down))
    finally:
        for p in (pa, pc, pc2, po, pd):
            p.free()
        for x in (w, w2, wd):
            x.destroy()


@pytest.mark.parametrize("entry,m,k,n,nd", [("multi", 520, 3072, 8448, 0), ("swiglu", 520, 3072, 8448, 0), ("down", 520, 1024, 6400, 8192),
                                               ("down", 520, 2048, 8448, 8448), ("multi", 1100, 1536, 3072, 0)])
def test_grouped_q6_K_prefill_rows_cross_in_steps(hipq, cr, entry, m, k, n, nd):
    """The calls of several weights: 512 rows and more cross in steps of 256, the last of up to 511, whatever a step's 256 rows
    alone would be formed in. At the first three sizes that would be parts of K where the whole call walks K whole, at the
    fourth the down projection of the whole call is formed in parts of K. A step's products take the whole call's parts, so
    that the outputs have the bits of the device-memory call."""
    import gpu_util as gu
    import torch

    def weight(j, rows, cols):
        few = cr.quantize_weights(cr.oracle(), "q6_K", synth.normal(9800 + j, (61, cols), 0.05)).reshape(61, -1)
        return capi.Weight("q6_K", rows, cols, np.ascontiguousarray(few[np.random.RandomState(j).randint(0, 61, rows)]))

    ws = [weight(0, n, k), weight(1, n, k)] + ([weight(2, nd, n)] if nd else [])
    a = synth.normal(9810 + m, (m, k))
    pa = _Pinned((m, k), a)
    shapes = [(m, n), (m, n)] if entry == "multi" else [(m, nd or n)]
    out = [_Pinned(x, np.nan) for x in shapes]
    dev = [torch.full(x, float("nan"), device="cuda") for x in shapes]

    def call(rows, res, **kw):
        if entry == "multi":
            capi.matmul_multi(ws, rows, m, res, **kw)
        else:
            (capi.mlp_swiglu if entry == "swiglu" else capi.mlp_swiglu_down)(*ws, rows, m, res[0], **kw)

    try:
        with capi.LaunchTiming(64) as t:
            call(gu.dev(a), dev, stream=gu.stream())
            torch.cuda.synchronize()
        in_parts = ["split" in name for name, _ in t.launches if name.startswith("gemm_q6k")]
        with capi.LaunchTiming(64) as t:
            call(pa.addr, [o.addr for o in out], mem=capi.MEM_HOST)
        steps = ["split" in name for name, _ in t.launches if name.startswith("gemm_q6k")]
        for o, d in zip(out, dev):
            assert np.array_equal(o.arr.view(np.uint32), d.cpu().numpy().view(np.uint32))
        assert len(in_parts) == len(ws) and steps == (m // 256) * in_parts, (in_parts, steps)
    finally:
        for x in [pa] + out:
            x.free()
        for w in ws:
            w.destroy()


@pytest.mark.parametrize("kind,m,k,ns", [
    ("q4_K", 8, 512, (1024,)), ("q4_K", 6, 256, (4099,)),       # 32 workgroups; 129, the last with three columns
    ("q4_K", 64, 256, (1030,)), ("q4_K", 4, 512, (384, 640, 31)),  # eight passes; three weights of a launch
    ("q4_0", 2, 1024, (512,)), ("q4_0", 16, 2048, (520,)),      # rows quantized by the kernel; 17 workgroups a pass
    ("q4_0", 3, 512, (600, 200, 300, 32)), ("q6_K", 16, 256, (33,)), ("q6_K", 5, 1024, (6001,)),
])
def test_calls_that_their_last_workgroup_ends(hipq, cr, kind, m, k, ns):
    """A few rows of host memory through the kernels of gemm_rows_*.hip: the last workgroup of the launch tells the host that
    the outputs are there. Launches of fewer workgroups than arrival counters, of no whole multiple of them, of several
    passes and weights; many calls one after the other, each with outputs of its own (a flag that came early would show the
    values of the call before). The device call's bits, page-locked and pageable."""
    ws = [capi.Weight(kind, n, k, cr.quantize_weights(cr.oracle(), kind, synth.normal(9700 + n, (n, k), 0.02))) for n in ns]
    a = synth.normal(9701 + m, (m, k))
    want = [_device_result(w, a) for w in ws] if len(ws) == 1 else None
    if want is None:
        import gpu_util as gu
        import torch
        out = [torch.empty((m, n), device="cuda") for n in ns]
        capi.matmul_multi(ws, gu.dev(a), m, out, stream=gu.stream())
        torch.cuda.synchronize()
        want = [o.cpu().numpy() for o in out]
    pa, pc = capi.host_alloc(m * k * 4), [capi.host_alloc(m * n * 4) for n in ns]
    try:
        a_pin = np.ctypeslib.as_array(ctypes.cast(pa, ctypes.POINTER(ctypes.c_float)), (m, k))
        c_pin = [np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), (m, n)) for p, n in zip(pc, ns)]
        c_page = [np.empty((m, n), np.float32) for n in ns]
        for rep in range(40):
            scale = np.float32(2.0 ** (rep % 5))  # powers of two: the outputs scale exactly
            a_pin[:] = a * scale
            pinned = rep % 4 != 3
            for c in c_pin + c_page:
                c[:] = np.nan
            outs = c_pin if pinned else c_page
            if len(ws) == 1:
                capi.matmul(ws[0], pa, m, pc[0] if pinned else c_page[0], mem=capi.MEM_HOST)
            else:
                capi.matmul_multi(ws, pa, m, pc if pinned else c_page, mem=capi.MEM_HOST)
            for got, ref in zip(outs, want):
                assert np.array_equal(got, ref * scale)
    finally:
        for p in [pa] + pc:
            capi.host_free(p)
        for w in ws:
            w.destroy()


def test_threads_in_turn_on_the_per_thread_stream(hipq, cr):
    """Two threads that share the handle hipStreamPerThread, call after call in turn: queues of their own, one set of arrival
    counters and one word, ordered by each call's return alone. The device call's bits, 129 and 32 workgroups."""
    import threading
    per_thread = 2  # hipStreamPerThread
    work = []
    for m, n, k in ((8, 4100, 256), (3, 1024, 512)):
        w = capi.Weight("q4_K", n, k, cr.quantize_weights(cr.oracle(), "q4_K", synth.normal(9800 + n, (n, k), 0.02)))
        a = synth.normal(9801 + n, (m, k))
        work.append((w, m, n, k, a, _device_result(w, a), capi.host_alloc(m * k * 4), capi.host_alloc(m * n * 4)))
    turn, failed = threading.Semaphore(1), []

    def calls(index):
        w, m, n, k, a, want, pa, pc = work[index]
        a_pin = np.ctypeslib.as_array(ctypes.cast(pa, ctypes.POINTER(ctypes.c_float)), (m, k))
        c_pin = np.ctypeslib.as_array(ctypes.cast(pc, ctypes.POINTER(ctypes.c_float)), (m, n))
        for rep in range(100):
            scale = np.float32(2.0 ** (rep % 5))
            with turn:
                a_pin[:] = a * scale
                c_pin[:] = np.nan
                capi.matmul(w, pa, m, pc, mem=capi.MEM_HOST, stream=per_thread)
                if not np.array_equal(c_pin, want * scale):
                    failed.append((index, rep))

    threads = [threading.Thread(target=calls, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    capi.stream_release(per_thread)
    for w, _, _, _, _, _, pa, pc in work:
        capi.host_free(pa)
        capi.host_free(pc)
        w.destroy()
    assert not failed


def test_a_streams_first_host_call_waits_for_no_other_stream(hipq, cr):
    """What a stream's first call on host memory sets up is made in order on that stream: work under way on the default stream,
    hundreds of milliseconds of it, is still under way when the call returns."""
    import torch
    m, n, k = 8, 2048, 512
    w = capi.Weight("q4_K", n, k, cr.quantize_weights(cr.oracle(), "q4_K", synth.normal(9900, (n, k), 0.02)))
    a = synth.normal(9901, (m, k))
    want = _device_result(w, a)
    pa, pc = capi.host_alloc(m * k * 4), capi.host_alloc(m * n * 4)
    try:
        np.ctypeslib.as_array(ctypes.cast(pa, ctypes.POINTER(ctypes.c_float)), (m, k))[:] = a
        c_pin = np.ctypeslib.as_array(ctypes.cast(pc, ctypes.POINTER(ctypes.c_float)), (m, n))
        x, y = (torch.ones((8192, 8192), device="cuda", dtype=torch.bfloat16) for _ in range(2))
        other, end = torch.cuda.Stream(), torch.cuda.Event()
        capi.matmul(w, pa, m, pc, mem=capi.MEM_HOST, stream=other.cuda_stream)
        capi.stream_release(other.cuda_stream)
        torch.mm(x, x, out=y)
        torch.cuda.synchronize()
        for _ in range(300):
            torch.mm(x, x, out=y)
        end.record()
        for _ in range(2):
            c_pin[:] = np.nan
            capi.matmul(w, pa, m, pc, mem=capi.MEM_HOST, stream=other.cuda_stream)
            assert np.array_equal(c_pin.view(np.uint32), want.view(np.uint32))
        assert not end.query()
        torch.cuda.synchronize()
        capi.stream_release(other.cuda_stream)
    finally:
        torch.cuda.synchronize()
        capi.host_free(pa)
        capi.host_free(pc)
        w.destroy()


@pytest.mark.parametrize("kind,rows,one_launch", [("q6_K", 16, True), ("q6_K", 24, False), ("q6_K", 40, False), ("q4_K", 64, True),
                                                  ("q4_K", 72, False), ("q4_0", 24, True)])
def test_only_a_launch_that_writes_all_outputs_ends_its_call(hipq, cr, kind, rows, one_launch):
    """Rows as products of their own in host memory: one launch up to 16 (Q6_K) and 64 rows (Q4_K), which tells the host itself;
    more rows take several, and a launch behind all of them ends the call. The device call's bits."""
    n, k = 4100, 512
    w = capi.Weight(kind, n, k, cr.quantize_weights(cr.oracle(), kind, synth.normal(9950 + rows, (n, k), 0.02)))
    a = synth.normal(9951, (rows, k))
    import gpu_util as gu
    import torch
    want = torch.empty((rows, n), device="cuda")
    with capi.LaunchTiming(64) as t:
        capi.matmul_each_row(w, gu.dev(a), rows, want, stream=gu.stream())
    torch.cuda.synchronize()
    form = ("gemm_rows_q40", "gemm_rows_q6k")  # host calls have a form of these kernels of their own
    assert all(name.endswith("false>") for name, _ in t.launches if name.startswith(form))
    pa, pc = capi.host_alloc(rows * k * 4), capi.host_alloc(rows * n * 4)
    try:
        np.ctypeslib.as_array(ctypes.cast(pa, ctypes.POINTER(ctypes.c_float)), (rows, k))[:] = a
        c_pin = np.ctypeslib.as_array(ctypes.cast(pc, ctypes.POINTER(ctypes.c_float)), (rows, n))
        c_pin[:] = np.nan
        with capi.LaunchTiming(64) as t:
            capi.matmul_each_row(w, pa, rows, pc, mem=capi.MEM_HOST, stream=gu.stream())
        assert np.array_equal(c_pin.view(np.uint32), want.cpu().numpy().view(np.uint32))
        names = [name for name, _ in t.launches]
        products = [x for x in names if x.startswith("gemm_rows_")]
        assert (len(products) == 1) == one_launch and (names[-1] != "signal_done_kernel") == one_launch, names
        assert all(x.endswith("true>" if one_launch else "false>") for x in products if x.startswith(form)), names
    finally:
        capi.host_free(pa)
        capi.host_free(pc)
        w.destroy()
