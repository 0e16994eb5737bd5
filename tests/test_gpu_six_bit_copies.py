"""The six-bit copy a Q4_0 weight gets at its first product of many rows (gemm_f6.hip): when it can be had, who may
read it, and what a call does without it. Every kernel of the format has the reference's bits, so the products are
compared bit for bit; which kernel ran is read from the launch log."""
import numpy as np
import pytest

from nntrainer_amd import capi, synth

pytestmark = pytest.mark.gpu


def _weight(n, k, seed):
    """A Q4_0 weight of random blocks with scales near 0.01, made on the device."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    blocks = torch.randint(0, 256, (n * k // 32, 18), generator=gen, device="cuda", dtype=torch.uint8)
    scales = torch.rand(n * k // 32, generator=gen, device="cuda").mul_(0.01).add_(0.005).half()
    blocks[:, :2] = scales.view(torch.uint8).view(-1, 2)
    torch.cuda.synchronize()
    return capi.Weight("q4_0", n, k, blocks, mem=capi.MEM_DEVICE)


def _kernels(call):
    """Runs call and names the kernels it launched."""
    with capi.LaunchTiming(64) as t:
        call()
    return [name.split("<")[0] for name, _ in t.launches]


def test_a_product_of_many_rows_on_a_full_device(hipq):
    """Where the copy's memory is refused the kernels that read the weight as stored take the call, and the refusal is
    not reported by a later launch; once there is memory the copy is made. 524288 x 2048: 872 MB."""
    import torch
    n, k, m = 524288, 2048, 65
    s = torch.cuda.current_stream().cuda_stream
    w = _weight(n, k, 1)
    a = torch.randn((m, k), device="cuda")
    want, got = (torch.full((m, n), float("nan"), device="cuda") for _ in range(2))
    # both paths' kernels and workspaces are there before the memory goes: the stored planes, and a copy of another weight
    capi.matmul_noalloc(w, a, m, want, stream=s)
    small = _weight(256, k, 2)
    capi.matmul(small, a, m, torch.empty((m, 256), device="cuda"), stream=s)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    hold = []
    try:
        for step, leave in ((1 << 33, 1 << 34), (1 << 30, 1 << 31), (1 << 25, 256 << 20)):
            while torch.cuda.mem_get_info()[0] - step > leave:
                hold.append(torch.empty(step, dtype=torch.uint8, device="cuda"))
        assert torch.cuda.mem_get_info()[0] < 300 << 20  # the copy takes 872 MB
        for _ in range(2):
            got.fill_(float("nan"))
            names = _kernels(lambda: capi.matmul(w, a, m, got, stream=s))
            torch.cuda.synchronize()
            assert "gemm_f6_kernel" not in names and torch.equal(got, want)
    finally:
        hold.clear()
        torch.cuda.empty_cache()
    got.fill_(float("nan"))
    names = _kernels(lambda: capi.matmul(w, a, m, got, stream=s))
    torch.cuda.synchronize()
    assert "gemm_f6_kernel" in names and torch.equal(got, want)
    w.destroy()
    small.destroy()


class _Graph:
    """What a call enqueues on a stream, captured: .nodes launches, .launch(stream) replays them."""

    def __init__(self, stream, call):
        import ctypes as C
        path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
        self.hip, self.graph, self.exec = C.CDLL(path), C.c_void_p(), C.c_void_p()
        s, n = C.c_void_p(stream), C.c_size_t()
        assert self.hip.hipStreamBeginCapture(s, 1) == 0  # thread-local
        try:
            call(stream)
        finally:
            assert self.hip.hipStreamEndCapture(s, C.byref(self.graph)) == 0
        assert self.hip.hipGraphGetNodes(self.graph, None, C.byref(n)) == 0
        assert self.hip.hipGraphInstantiate(C.byref(self.exec), self.graph, None, None, C.c_size_t(0)) == 0
        self.nodes = n.value

    def launch(self, stream):
        import ctypes as C
        assert self.hip.hipGraphLaunch(self.exec, C.c_void_p(stream)) == 0

    def destroy(self):
        self.hip.hipGraphExecDestroy(self.exec)
        self.hip.hipGraphDestroy(self.graph)


N, K, M = 130, 96, 200  # a K that the int8 GEMM does not take: without the copy a call is 25 eight-row passes
WITH_COPY, WITHOUT = 2, 26  # launches of a call, the quantizer among them


def _case(seed):
    import torch
    w, other = _weight(N, K, seed), _weight(N, K, seed + 1)
    a = torch.randn((M, K), device="cuda")
    want = torch.full((M, N), float("nan"), device="cuda")
    capi.matmul_noalloc(w, a, M, want, stream=torch.cuda.current_stream().cuda_stream)
    streams = [torch.cuda.Stream() for _ in range(2)]
    for st in streams:  # the workspaces, by a weight of its own
        capi.matmul(other, a, M, torch.empty((M, N), device="cuda"), stream=st.cuda_stream)
    torch.cuda.synchronize()
    return w, other, a, want, streams


def _done(w, other, streams):
    import torch
    torch.cuda.synchronize()
    for st in streams:
        capi.stream_release(st.cuda_stream)
    w.destroy()
    other.destroy()


def test_a_graph_captured_on_another_stream_reads_the_complete_copy(hipq):
    """A weight warmed up on one stream, its product captured on another: the graph has the six-bit kernel, and every
    replay, with eager work between, the bits of the stored weights' kernels."""
    import torch
    w, other, a, want, (first, second) = _case(10)
    got, eager = (torch.full((M, N), float("nan"), device="cuda") for _ in range(2))
    capi.matmul(w, a, M, eager, stream=first.cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(eager, want)
    graph = _Graph(second.cuda_stream, lambda s: capi.matmul(w, a, M, got, stream=s))
    assert graph.nodes == WITH_COPY
    for _ in range(4):
        got.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.launch(second.cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        capi.matmul(w, a, M, eager, stream=second.cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(eager, want)
    graph.destroy()
    _done(w, other, (first, second))


def test_a_copy_that_is_not_complete_is_read_on_its_own_stream_only(hipq):
    """The call that makes the copy waits behind 300 ms of other work on its stream. A second call on that stream reads
    the copy; one on another stream, and one captured into a graph, does not and does not wait; once the copy is
    complete all do. The same bits everywhere."""
    import torch
    w, other, a, want, (first, second) = _case(20)
    outs = [torch.full((M, N), float("nan"), device="cuda") for _ in range(5)]
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        torch.cuda._sleep(int(0.3 * 2.0e9))
    capi.matmul(w, a, M, outs[0], stream=first.cuda_stream)
    capi.matmul(w, a, M, outs[1], stream=first.cuda_stream)
    capi.matmul(w, a, M, outs[2], stream=second.cuda_stream)
    pending = _Graph(second.cuda_stream, lambda s: capi.matmul(w, a, M, outs[3], stream=s))
    own = _Graph(first.cuda_stream, lambda s: capi.matmul(w, a, M, outs[4], stream=s))
    second.synchronize()
    still = not first.query()  # else this host took longer than the work in front: the results alone are checked
    assert torch.equal(outs[2], want)
    torch.cuda.synchronize()
    assert not still or (pending.nodes == WITHOUT and own.nodes == WITHOUT)
    pending.launch(second.cuda_stream)
    own.launch(first.cuda_stream)
    torch.cuda.synchronize()
    for got in outs:
        assert torch.equal(got, want)
    for st in (first, second):
        after = _Graph(st.cuda_stream, lambda s: capi.matmul(w, a, M, outs[3], stream=s))
        outs[3].fill_(float("nan"))
        torch.cuda.synchronize()
        after.launch(st.cuda_stream)
        torch.cuda.synchronize()
        assert after.nodes == WITH_COPY and torch.equal(outs[3], want)
        after.destroy()
    pending.destroy()
    own.destroy()
    _done(w, other, (first, second))


def test_two_threads_make_and_read_the_copies_of_the_same_weights(hipq):
    """Several weights, each thread on its own stream and in its own order, singly and as a group, without waiting
    between: whoever comes first makes a weight's copy."""
    import threading
    import torch
    w, other, a, want, streams = _case(30)
    for rep in range(4):
        ws = [_weight(N + 32 * i, K, 31 + i) for i in range(6)]
        wants = [torch.full((M, x.n), float("nan"), device="cuda") for x in ws]
        for x, o in zip(ws, wants):
            capi.matmul_noalloc(x, a, M, o, stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        outs = [[torch.full((M, x.n), float("nan"), device="cuda") for x in ws] for _ in range(2)]
        torch.cuda.synchronize()
        failed = []

        def work(t):
            try:
                order = list(range(6))[::1 if t else -1]
                for _ in range(3):
                    capi.matmul_multi([ws[i] for i in order[:3]], a, M, [outs[t][i] for i in order[:3]], stream=streams[t].cuda_stream)
                    for i in order[3:]:
                        capi.matmul(ws[i], a, M, outs[t][i], stream=streams[t].cuda_stream)
                streams[t].synchronize()
            except Exception as e:
                failed.append(e)
        threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not failed, failed
        for t in range(2):
            for got, o in zip(outs[t], wants):
                assert torch.equal(got, o)
        for x in ws:
            x.destroy()
    _done(w, other, streams)


def test_copies_share_blocks_of_memory_and_give_them_back(hipq):
    """Weights come and go in a seeded order, sizes from one tile to a copy with a block of its own, singly and in groups
    of up to nine (three launches of copies): every product has the bits of the stored weights' kernels, first and
    second, and when the last weight is gone so is all but one block of memory."""
    import random
    import torch
    rng = random.Random(5)
    s = torch.cuda.current_stream().cuda_stream
    m, k = 70, 1056
    a = torch.randn((m, k), device="cuda")
    big = 40000  # 40000 x 1280 (K padded) of 0.8125 bytes: 42 MB
    capi.matmul_noalloc(_weight(64, k, 90), a, m, torch.empty((m, 64), device="cuda"), stream=s)
    live = [_weight(64, k, 91)]
    capi.matmul(live[0], a, m, torch.empty((m, 64), device="cuda"), stream=s)  # the first block
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.mem_get_info()[0]
    for step in range(40):
        if len(live) > 1 and (rng.random() < 0.45 or step > 34):
            for w in [live.pop(rng.randrange(len(live))) for _ in range(min(len(live), rng.randint(1, 6)))]:
                w.destroy()
            continue
        ws = [_weight(big if rng.random() < 0.1 else rng.choice((1, 33, 2000, 9000, 12000)), k, 100 + 10 * step + i)
              for i in range(rng.randint(1, 9))]
        group = ws + rng.sample(live, min(2, len(live))) + ws[:1]
        wants = [torch.full((m, w.n), float("nan"), device="cuda") for w in group]
        gots = [torch.full((m, w.n), float("nan"), device="cuda") for w in group]
        for w, o in zip(ws, wants):
            capi.matmul_noalloc(w, a, m, o, stream=s)  # no copy yet
        for w, o in zip(group[len(ws):], wants[len(ws):]):
            capi.matmul_noalloc(w, a, m, o, stream=s)
        for _ in range(2):
            capi.matmul_multi(group, a, m, gots, stream=s)
            torch.cuda.synchronize()
            for got, o in zip(gots, wants):
                assert torch.equal(got, o), step
        live += ws
    for w in live:
        w.destroy()
    del ws, group, wants, gots, o, got
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    assert torch.cuda.mem_get_info()[0] >= before - (66 << 20)
