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
    not reported by a later launch; once there is memory the copy is made. 131072 x 2048: 218 MB."""
    import torch
    n, k, m = 131072, 2048, 65
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
        for step, leave in ((1 << 33, 1 << 34), (1 << 30, 1 << 31), (1 << 25, 150 << 20)):
            while torch.cuda.mem_get_info()[0] - step > leave:
                hold.append(torch.empty(step, dtype=torch.uint8, device="cuda"))
        assert torch.cuda.mem_get_info()[0] < 200 << 20
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
