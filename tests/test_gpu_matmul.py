"""GPU parity: fp32 outputs of the quantized matmul (decode GEMV and prefill GEMM)
against the oracle on the same seeded inputs, through the C ABI.

Bar: max|gpu - ref| / max|ref| <= 1e-4 per matrix (only the order of the fp32
additions may differ; integer inner sums are exact on both sides)."""
import numpy as np
import pytest

from nntrainer_amd import capi, synth

pytestmark = pytest.mark.gpu

KINDS = ["q4_0", "q4_K", "q6_K"]


def _weights(cr, kind, n, k, seed):
    w = synth.normal(seed, (n, k), 0.02)
    return cr.quantize_weights(cr.oracle(), kind, w)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,k", [(256, 256), (512, 1024), (1000, 768), (4096, 4096), (768, 2048),
                                 (130, 8192), (64, 12288)])
def test_gemv_matches_oracle(hipq, cr, kind, n, k):
    import gpu_util as gu
    if kind != "q4_0" and k % 256:
        pytest.skip("K must be a multiple of 256")
    blocks = _weights(cr, kind, n, k, seed=100 + n)
    a = synth.normal(200 + k, (1, k))
    ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
    w = capi.Weight(kind, n, k, blocks)
    got = gu.gpu_matmul(w, a)
    w.destroy()
    assert not np.isnan(got).any()
    assert gu.rel_err(got, ref) <= gu.TOL, gu.rel_err(got, ref)
    # the decode path reproduces the reference's fp32 evaluation order: same bits
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
        "%d of %d outputs differ in bits" % ((got.view(np.uint32) != ref.view(np.uint32)).sum(), got.size)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,k", [(6150, 4096), (8200, 4096), (12290, 4096), (2050, 3072), (1024, 3072),
                                 (3000, 2304), (2100, 2560), (9000, 2048), (33000, 4096), (33000, 2048),
                                 (1000, 1024), (40000, 1024)])
def test_single_row_against_the_instances_by_row_length(hipq, cr, kind, n, k):
    """One row against shapes chosen by what the library picks for them: the kernels with the row length as
    a constant (1024, 2048, 3072, 4096) and the ones that take any length (2304, 2560), last workgroups that
    hang over the matrix's end (6150, 8200, 12290), the kernel behind the quantizer's launch (33000 and 40000
    columns). Same bits as the reference's row product."""
    import gpu_util as gu
    blocks = _weights(cr, kind, n, k, seed=900 + n % 97)
    a = synth.normal(950 + k % 89, (1, k))
    ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
    w = capi.Weight(kind, n, k, blocks)
    got = gu.gpu_matmul(w, a)
    w.destroy()
    assert not np.isnan(got).any()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
        "%d of %d outputs differ in bits" % ((got.view(np.uint32) != ref.view(np.uint32)).sum(), got.size)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,k", [
    # rows within one chunk: at, above and below whole steps of the 16, 32 and 64 lanes a row, and of the sums' batches
    (100, 512), (6144, 768), (70, 1280), (1024, 1792), (1025, 2304), (2049, 2816), (2051, 3328), (3000, 3840), (4100, 3584),
    # rows that a workgroup's wavefronts share, quantized in the kernel: one to four rows a wavefront, parts of unequal
    # length, the longest row
    (3, 4352), (1024, 4608), (1025, 6400), (1030, 8192), (4096, 16384), (37, 12544), (8192, 4352),
    # the same behind the quantizer's launch: more rows, rows longer than one pass of a workgroup quantizes
    (8193, 4352), (9, 16640), (70, 32768),
    # longer than 32768 (Q6_K: 65536): walked in chunks
    (5, 33024),
    # the wide matrices behind the quantizer's launch
    (32769, 512), (32771, 1792), (32770, 2816), (32773, 3840)])
def test_single_row_by_length_and_rows(hipq, cr, kind, n, k):
    """One row against matrices around the lines of the GEMV's dispatch (lanes a row, rows a wavefront, steps of a lane,
    parts of a long row). Same bits as the reference's row product; the weights are random blocks of few distinct rows."""
    import gpu_util as gu
    few = _weights(cr, kind, min(n, 61), k, seed=2000 + n % 97)
    rows = np.random.RandomState(n).randint(0, min(n, 61), n)
    blocks = np.ascontiguousarray(few.reshape(min(n, 61), -1)[rows])
    a = synth.normal(2100 + k % 89, (1, k))
    ref = cr.gemm(cr.oracle(), kind, a, few, min(n, 61))[:, rows]
    w = capi.Weight(kind, n, k, blocks)
    got = gu.gpu_matmul(w, a)
    w.destroy()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
        "%d of %d outputs differ in bits" % ((got.view(np.uint32) != ref.view(np.uint32)).sum(), got.size)


@pytest.mark.parametrize("k", [32, 800, 2336, 4128, 6112, 16352, 33056])
def test_single_q4_0_row_of_whole_blocks_only(hipq, cr, k):
    """Rows of whole blocks of 32 that end inside a batch of the sums' records and inside a part of a long row."""
    import gpu_util as gu
    for n in (33, 2100):
        few = _weights(cr, "q4_0", 33, k, seed=2200 + k % 97)
        rows = np.random.RandomState(n).randint(0, 33, n)
        a = synth.normal(2300 + k % 89, (1, k))
        ref = cr.gemm(cr.oracle(), "q4_0", a, few, 33)[:, rows]
        w = capi.Weight("q4_0", n, k, np.ascontiguousarray(few.reshape(33, -1)[rows]))
        got = gu.gpu_matmul(w, a)
        w.destroy()
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (n, k)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,k", [(770, 1792), (1024, 2304), (2050, 2816), (2048, 3072), (600, 3584), (2500, 3840)])
def test_gated_pair_of_one_row_by_length_and_rows(hipq, cr, kind, n, k):
    """mlp_swiglu on one row takes the same forms with two matrices a wavefront: its sums have the bits of the two single
    products, seen through the activation as numpy forms it from them (a few units in the last place of its exponential)."""
    import gpu_util as gu
    a = synth.normal(2400 + k % 89, (1, k))
    few = [_weights(cr, kind, 41, k, seed=2500 + i) for i in range(2)]
    rows = [np.random.RandomState(n + i).randint(0, 41, n) for i in range(2)]
    y, z = (cr.gemm(cr.oracle(), kind, a, few[i], 41)[0, rows[i]] for i in range(2))
    ws = [capi.Weight(kind, n, k, np.ascontiguousarray(few[i].reshape(41, -1)[rows[i]])) for i in range(2)]
    da, out = gu.dev(a), gu.dev(np.full((1, n), np.nan, np.float32))
    capi.mlp_swiglu(ws[0], ws[1], da, 1, out, stream=gu.stream())
    got = out.cpu().numpy()[0].astype(np.float64)
    for w in ws:
        w.destroy()
    want = y.astype(np.float64) / (1 + np.exp(-y.astype(np.float64))) * z.astype(np.float64)
    # exp, sum, quotient and product: under eight roundings of 2^-24 relative
    assert (np.abs(got - want) <= 8 * 2.0 ** -24 * np.abs(want) + 1e-30).all(), np.abs(got / want - 1).max()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m", [2, 3, 4, 5, 7, 8])
def test_small_m_matches_oracle(hipq, cr, kind, m):
    """M = 2..8 runs the multi-row GEMV; rows below 4*(M/4) of a Q4_K matmul must be
    quantized with the 4-row rule, the rest with the row rule."""
    import gpu_util as gu
    n, k = 512, 1024
    blocks = _weights(cr, kind, n, k, seed=31)
    a = synth.normal(300 + m, (m, k))
    ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
    w = capi.Weight(kind, n, k, blocks)
    got = gu.gpu_matmul(w, a)
    w.destroy()
    assert gu.rel_err(got, ref) <= gu.TOL, gu.rel_err(got, ref)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m,n,k", [(3, 2304, 2048), (4, 2050, 4096), (5, 2056, 2048), (8, 4100, 2048),
                                   (7, 12288, 2048), (3, 8200, 1024), (4, 8195, 2048), (6, 1100, 768),
                                   (8, 1024, 256), (5, 3000, 4096), (8, 1030, 8192), (6, 1024, 5376),
                                   (4, 4100, 1280), (9, 1100, 1024), (14, 2048, 512), (16, 1024, 2048),
                                   (11, 4000, 4096), (6, 32768, 1024), (8, 8200, 4096), (24, 4096, 2048),
                                   (64, 2048, 2048), (33, 1056, 4096), (2, 16400, 1024), (4, 6150, 4096),
                                   (3, 12290, 4096), (4, 4100, 4096), (2, 33000, 2048)])
def test_small_m_on_large_matrices_matches_oracle(hipq, cr, kind, m, n, k):
    """Three to sixteen rows against larger matrices, where Q4_K leaves the GEMV engine (and, from
    nine rows, the prefill GEMM) for the matrix-core kernel of gemm_rows_q4k.hip (five rows and
    more from 1024 columns up, four from 4096 or, with rows of 4096, 6144, three from 8192 or 12288,
    two against 16384 rows of 1024; more than eight rows as passes
    of eight side by side in one launch, up to 64 rows where the product is small, the later
    passes with fewer rows under the 4-row rule or none): rows under the reference's
    4-row rule and under its row rule in one call
    (6 = 4 + 2), one to 32 super-blocks a row (a round of four wavefronts partly idle, a single
    round, rows longer than the GEMV engine's 4096-weight chunk), column counts that end inside
    a 32-column tile; five to eight rows against 2^25 weights and more, where Q4_0 takes its
    matrix-core GEMM. Same bits as the reference, for all three formats."""
    import gpu_util as gu
    blocks = _weights(cr, kind, n, k, seed=700 + n)
    a = synth.normal(701 + k + m, (m, k))
    ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
    w = capi.Weight(kind, n, k, blocks)
    got = gu.gpu_matmul(w, a)
    w.destroy()
    engine_rows = 2 if n * k >= 2 ** 28 else 4 if n * k >= 2 ** 25 else 8 if n * k >= 2 ** 24 else 16
    if kind == "q6_K" and m > engine_rows:
        # Q6_K leaves the GEMV engine earlier on large matrices (the matrix cores are faster there)
        assert gu.rel_err(got, ref) <= gu.TOL, gu.rel_err(got, ref)
        return
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
        "%d of %d outputs differ in bits" % ((got.view(np.uint32) != ref.view(np.uint32)).sum(), got.size)


@pytest.mark.parametrize("m,n,k", [(1, 65553, 1024), (1, 65536, 256), (2, 12300, 512), (3, 6150, 768),
                                   (2, 600, 1024), (3, 16000, 512), (4, 2050, 768), (2, 16500, 1024),
                                   (6, 1030, 1024), (8, 2048, 512), (5, 520, 768),
                                   (4, 6144, 1024), (5, 3100, 1280), (7, 3072, 256), (9, 640, 256),
                                   (12, 600, 2304), (16, 513, 1024), (17, 520, 5120), (40, 1500, 1024),
                                   (64, 4096, 256), (57, 2050, 1280)])
def test_q4_0_few_rows_on_the_matrix_cores_match_oracle(hipq, cr, m, n, k):
    """Q4_0 with a few rows where gemm_rows_q40.hip takes them (one row against a wide matrix of
    short rows, two rows from 12288 columns of 1024 or 32768 longer ones, three and four from 6144,
    two to eight from 512 where the kernel quantizes the rows itself, five to eight from 3072,
    nine to sixteen from 512, up to 64 while the launch stays small): one to eight passes, one to
    five rounds of 32 blocks with the last one partly or wholly one wavefront's, column counts
    that end inside a 32-column tile. Same bits as the reference."""
    import gpu_util as gu
    blocks = _weights(cr, "q4_0", n, k, seed=1300 + m)
    a = synth.normal(1301 + k + m, (m, k))
    ref = cr.gemm(cr.oracle(), "q4_0", a, blocks, n)
    w = capi.Weight("q4_0", n, k, blocks)
    got = gu.gpu_matmul(w, a)
    w.destroy()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
        "%d of %d outputs differ in bits" % ((got.view(np.uint32) != ref.view(np.uint32)).sum(), got.size)


@pytest.mark.parametrize("m,n,k", [(65, 33, 32), (96, 128, 256), (97, 130, 544), (129, 1000, 768), (9, 300, 96),
                                   (31, 260, 1056), (200, 257, 2080), (2100, 1030, 288)])
def test_q4_0_on_six_bit_operands_matches_oracle(hipq, cr, m, n, k):
    """Q4_0 through gemm_f6.hip: row counts around the 32-row tile and the quantizer's 64, columns that end inside a
    tile and inside a workgroup's four, one to nine chunks of 256 of K with the last one whole, one block and three,
    and a launch of more than 512 workgroups. Activations with every 8-bit value. Same bits as the reference; a second
    call after another product of the stream's workspace."""
    import gpu_util as gu
    blocks = _weights(cr, "q4_0", n, k, seed=1400 + m)
    a = synth.normal(1401 + k + m, (m, k))
    ramp = (np.arange(k, dtype=np.float32) % 256 - 127.5) / 127.5
    a[::7] = ramp * np.abs(a[::7, :1])  # rows whose blocks run through the quantizer's range
    a[3::11, ::5] = 0.0
    ref = cr.gemm(cr.oracle(), "q4_0", a, blocks, n)
    w = capi.Weight("q4_0", n, k, blocks)
    for rep in range(2):
        got = gu.gpu_matmul(w, a)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
            "%d of %d outputs differ in bits" % ((got.view(np.uint32) != ref.view(np.uint32)).sum(), got.size)
        gu.gpu_matmul(w, synth.normal(rep, (70, k)))
    w.destroy()


@pytest.mark.parametrize("m,ns,k", [(128, (4096,), 288), (97, (4097,), 544), (129, (4000,), 256), (70, (33, 130, 64, 31), 800),
                                    (160, (1000, 2072), 288), (65, (64, 1, 65), 32), (512, (4096,), 256)])
def test_q4_0_on_six_bit_operands_with_few_tiles(hipq, cr, m, ns, k):
    """gemm_f6.hip with few tiles, where two wavefronts share one, each with the sums of half of its rows, and right above
    (f6_alone), alone and several weights a launch: columns that end inside the 64 of a workgroup and in front of
    its second tile, rows that end inside the upper and the lower half. Same bits as the reference."""
    import gpu_util as gu
    import torch
    blocks = [_weights(cr, "q4_0", n, k, seed=1500 + n) for n in ns]
    a = synth.normal(1501 + k + m, (m, k))
    w = [capi.Weight("q4_0", n, k, b) for n, b in zip(ns, blocks)]
    da = gu.dev(a)
    out = [torch.full((m, n + 3), float("nan"), device="cuda") for n in ns]
    capi.matmul_multi(w, da, m, out, ldc=[n + 3 for n in ns], stream=gu.stream())
    torch.cuda.synchronize()
    for x, n, b, o in zip(w, ns, blocks, out):
        ref, got = cr.gemm(cr.oracle(), "q4_0", a, b, n), o.cpu().numpy()
        assert np.array_equal(np.ascontiguousarray(got[:, :n]).view(np.uint32), ref.view(np.uint32))
        assert np.isnan(got[:, n:]).all()
        assert np.array_equal(gu.gpu_matmul(x, a).view(np.uint32), ref.view(np.uint32))
        x.destroy()


@pytest.mark.parametrize("m,n,form", [
    (512, 1024, "<3, true, 8>"), (513, 1024, "<3, true, 16>"), (525, 865, "<3, true, 16>"), (128, 4096, "<3, true, 8>"),
    (128, 4097, "<3, true, 16>"), (33, 8192, "<3, true, 8>"), (33, 8193, "<3, true, 16>"), (1024, 512, "<3, true, 8>"),
    (1025, 512, "<3, false, 16>"), (1024, 513, "<3, true, 16>"), (1300, 300, "<3, true, 8>"), (4096, 128, "<3, true, 8>"),
    (4097, 128, "<3, false, 16>"), (512, 2048, "<3, true, 16>"), (513, 2048, "<3, false, 16>"), (512, 2049, "<3, false, 16>"),
    (512, 4096, "<3, false, 16>"), (512, 4097, "<1, false, 16>")])
def test_q4_0_tile_forms_by_an_xcds_workgroups(hipq, cr, m, n, form):
    """gemm_f6.hip: two wavefronts a tile, and the sums between the matrix instructions, where every workgroup has a CU of its own: an
    XCD's eighth of the workgroup columns, with all row tiles, against its 32 CUs, not their total (up to eight columns of two
    tiles are one an XCD however many rows there are). Both sides of the lines, the reference's bits."""
    import gpu_util as gu
    k = 64
    blocks = _weights(cr, "q4_0", n, k, seed=1600 + n)
    a = synth.normal(1601 + m, (m, k))
    w = capi.Weight("q4_0", n, k, blocks)
    gu.gpu_matmul(w, a)  # makes the six-bit copy
    with capi.LaunchTiming(16) as t:
        got = gu.gpu_matmul(w, a)
    assert [name for name, _ in t.launches if name.startswith("gemm_f6_kernel")] == ["gemm_f6_kernel" + form]
    assert np.array_equal(got.view(np.uint32), cr.gemm(cr.oracle(), "q4_0", a, blocks, n).view(np.uint32))
    w.destroy()


@pytest.mark.parametrize("m,n,form", [(512, 1024, "<3, true, "), (513, 1024, "<3, false, "), (512, 1056, "<3, false, "),
                                      (1024, 1024, "<3, false, "), (1025, 1024, "<1, false, ")])
def test_q4_0_gated_tile_forms_by_an_xcds_workgroups(hipq, cr, m, n, form):
    """The gated pair keeps to the same lines; its result as rows and as the down projection's operand."""
    import gpu_util as gu
    import torch
    k, nd = 64, 64
    ws = [capi.Weight("q4_0", r, c, _weights(cr, "q4_0", r, c, seed=1700 + i)) for i, (r, c) in enumerate([(n, k), (n, k), (nd, n)])]
    a = synth.normal(1701 + m, (m, k))
    da, h, out, two = gu.dev(a), torch.empty((m, n), device="cuda"), *(torch.empty((m, nd), device="cuda") for _ in range(2))
    for _ in range(2):  # the first calls make the six-bit copies
        with capi.LaunchTiming(32) as t:
            capi.mlp_swiglu(ws[0], ws[1], da, m, h, stream=gu.stream())
            capi.mlp_swiglu_down(*ws, da, m, out, stream=gu.stream())
        torch.cuda.synchronize()
    assert [name for name, _ in t.launches if "gated" in name] == ["gemm_f6_gated_kernel%s%s>" % (form, q) for q in ("false", "true")]
    y, z = gu.gpu_matmul(ws[0], a), gu.gpu_matmul(ws[1], a)
    ref = cr.swiglu(y, z)
    assert np.abs(h.cpu().numpy() - ref).max() <= 1e-6 * np.abs(ref).max()  # the device's expf against the host's
    capi.matmul(ws[2], h, m, two, stream=gu.stream())
    torch.cuda.synchronize()
    assert torch.equal(out, two)
    for w in ws:
        w.destroy()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,k", [(32800, 1024), (33000, 512), (40010, 256), (32768, 768), (50000, 1280)])
def test_single_row_against_wide_matrices_of_short_rows(hipq, cr, kind, n, k):
    """One row against 32768 columns or more with rows of fewer than 64 load units: Q4_0 and Q4_K
    stream them sixteen lanes a row, eight rows a group and two or four groups a wavefront with the
    next group's loads in flight (Q6_K keeps the plain kernel); column counts that end inside a
    group and inside a workgroup's share. Same bits as the reference."""
    import gpu_util as gu
    blocks = _weights(cr, kind, n, k, seed=1600 + k)
    a = synth.normal(1601 + n, (1, k))
    ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
    w = capi.Weight(kind, n, k, blocks)
    got = gu.gpu_matmul(w, a)
    w.destroy()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
        "%d of %d outputs differ in bits" % ((got.view(np.uint32) != ref.view(np.uint32)).sum(), got.size)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m,n,k", [(1, 8200, 12288), (3, 200, 8192), (8, 520, 9216), (1, 96, 20480),
                                   (5, 64, 4352)])
def test_rows_longer_than_one_chunk_match_oracle(hipq, cr, kind, m, n, k):
    """K above 4096 runs the GEMV instance that keeps the next chunk's weights in flight while
    the current chunk is computed: two, three and five chunks, a last chunk of 256, every group
    size the row count selects, one to eight activation rows. Same bits as the reference."""
    import gpu_util as gu
    blocks = _weights(cr, kind, n, k, seed=900 + n)
    a = synth.normal(901 + k + m, (m, k))
    ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
    w = capi.Weight(kind, n, k, blocks)
    got = gu.gpu_matmul(w, a)
    w.destroy()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
        "%d of %d outputs differ in bits" % ((got.view(np.uint32) != ref.view(np.uint32)).sum(), got.size)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m,n,k", [(16, 256, 256), (64, 512, 1024), (130, 384, 512), (457, 512, 512),
                                   (459, 512, 512), (512, 1024, 2048)])
def test_gemm_matches_oracle(hipq, cr, kind, m, n, k):
    """Prefill shapes, including M % 4 != 0 (the reference's leftover-row path,
    unittest_nntrainer_cpu_backend.cpp:457-515 uses M = 457, 458, 459) and tiles that
    do not divide M or N."""
    import gpu_util as gu
    blocks = _weights(cr, kind, n, k, seed=41 + m)
    a = synth.normal(400 + m, (m, k))
    ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
    w = capi.Weight(kind, n, k, blocks)
    got = gu.gpu_matmul(w, a)
    w.destroy()
    assert not np.isnan(got).any()
    assert gu.rel_err(got, ref) <= gu.TOL, gu.rel_err(got, ref)
    if kind == "q4_0":
        # Q4_0 (one fma per 32-block, in block order) reproduces the reference's fp32 order:
        # same bits, so a decoder's prefill cannot drift from the CPU leg. The matrix-core
        # GEMMs of the K-formats (two int8 planes per product) do not claim that.
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
            "%d of %d outputs differ in bits" % ((got.view(np.uint32) != ref.view(np.uint32)).sum(), got.size)


@pytest.mark.parametrize("m,n,k", [(17, 128, 256), (33, 200, 768), (64, 96, 1024), (100, 1000, 512),
                                   (512, 4096, 4096), (1100, 8192, 512), (12, 8192, 4096)])
def test_q6_K_gemm_matches_oracle(hipq, cr, m, n, k):
    """The Q6_K prefill product on the matrix cores: one and three super-blocks per row,
    N not a multiple of the 32-row weight tiles or of the 128-column workgroup tiles, M not a
    multiple of the tile heights, a shape that takes the 128-row tiles, the size of a
    Q6_K FC of a 4096-wide model, and twelve rows against a matrix of 2^25 weights (from that
    size on more than four rows leave the GEMV engine). Four rows keep the GEMV engine and the
    reference's bits at every size here."""
    import gpu_util as gu
    blocks = _weights(cr, "q6_K", n, k, seed=61 + m)
    a = synth.normal(600 + m, (m, k))
    a[0, :] = 0.0                      # a row of zero scales
    a[m - 1, 3] = 40.0                 # a row whose scale is set by one value
    ref = cr.gemm(cr.oracle(), "q6_K", a, blocks, n)
    w = capi.Weight("q6_K", n, k, blocks)
    got = gu.gpu_matmul(w, a)
    again = gu.gpu_matmul(w, a)        # the weight's tile copy exists now
    few = gu.gpu_matmul(w, a[:4])
    w.destroy()
    assert not np.isnan(got).any()
    assert gu.rel_err(got, ref) <= gu.TOL, gu.rel_err(got, ref)
    assert np.array_equal(got, again)
    assert np.array_equal(few.view(np.uint32), ref[:4].view(np.uint32))
    # per row as well: a row of small outputs must not hide behind the matrix maximum
    scale = np.abs(ref).max(axis=1)
    rows = scale > 0
    assert (np.abs(got - ref).max(axis=1)[rows] / scale[rows]).max() <= gu.TOL


def test_gemm_random_shapes_all_formats(hipq, cr):
    """Prefill products at shapes drawn from a seeded generator: N from 1 upward (narrower than a
    weight tile, between tile sizes), M between the GEMV limit and a few tiles, K one to five
    super-blocks. Every kernel's edge handling (padding rows and columns, odd super-block counts,
    both tile heights) is on some draw; the bar is the one of the fixed shapes."""
    import gpu_util as gu
    rng = np.random.RandomState(20240611)
    for case in range(24):
        kind = KINDS[case % 3]
        m = int(rng.choice([9, 17, 31, 64, 65, 127, 130, 257, 300]))
        n = int(rng.choice([1, 7, 31, 33, 100, 128, 129, 640, 1000, 4100]))
        k = 256 * int(rng.randint(1, 6))
        blocks = _weights(cr, kind, n, k, seed=500 + case)
        a = synth.normal(700 + case, (m, k))
        ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
        w = capi.Weight(kind, n, k, blocks)
        got = gu.gpu_matmul(w, a)
        w.destroy()
        assert not np.isnan(got).any(), (kind, m, n, k)
        assert gu.rel_err(got, ref) <= gu.TOL, (kind, m, n, k, gu.rel_err(got, ref))
        if kind == "q4_0":
            assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (kind, m, n, k)


@pytest.mark.parametrize("kind", ["q4_K", "q6_K"])
@pytest.mark.parametrize("m,n,k", [(17, 512, 2048), (40, 1000, 2304), (64, 4100, 4096), (100, 640, 3072),
                                   (128, 1536, 2048), (33, 1001, 2048)])
def test_k_format_gemm_in_parts_of_k(hipq, cr, kind, m, n, k):
    """Few tiles (up to 128 rows against a few thousand columns): once the weight has its tile copy
    the Q4_K and Q6_K prefill products are formed in parts of K that run side by side and are added in
    ascending order (nine super-blocks split 5 + 4, sixteen into four and eight parts). The first
    call, which makes the copy, and the following ones have the same bits, within 1e-4 of the
    reference; a strided output keeps its padding; N not a multiple of four likewise."""
    import gpu_util as gu
    import torch
    blocks = _weights(cr, kind, n, k, seed=330 + m)
    a = synth.normal(331 + m, (m, k))
    ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
    w = capi.Weight(kind, n, k, blocks)
    try:
        first = gu.gpu_matmul(w, a)
        assert gu.rel_err(first, ref) <= gu.TOL, gu.rel_err(first, ref)
        ldc = n + 12
        dc = torch.full((m, ldc), float("nan"), device="cuda")
        capi.matmul(w, gu.dev(a), m, dc, ldc=ldc, stream=gu.stream())
        torch.cuda.synchronize()
        got = dc[:, :n].cpu().numpy()
        assert not np.isnan(got).any()
        assert gu.rel_err(got, ref) <= gu.TOL, gu.rel_err(got, ref)
        assert torch.isnan(dc[:, n:]).all(), "the call wrote between the rows of C"
        assert np.array_equal(got, first), "the first call differs from the second"
        scale = np.abs(ref).max(axis=1)
        assert (np.abs(got - ref).max(axis=1) / scale).max() <= gu.TOL
        again = torch.full((m, n), float("nan"), device="cuda")
        capi.matmul_noalloc(w, gu.dev(a), m, again, stream=gu.stream())
        torch.cuda.synchronize()
        assert np.array_equal(again.cpu().numpy(), got), "the allocation-free call differs"
    finally:
        w.destroy()


@pytest.mark.parametrize("kind,m,n,k", [("q4_K", 700, 3000, 8192), ("q6_K", 700, 3000, 8192), ("q6_K", 520, 2052, 6144),
                                        ("q4_K", 400, 4096, 6400), ("q6_K", 200, 1000, 2304)])
def test_k_format_gemm_in_parts_of_k_by_tile_height(hipq, cr, kind, m, n, k):
    """Products that the plan of tile height and parts forms in parts of K beyond 128 rows: 128-row tiles in three parts of
    11, 11 and 10 super-blocks and in six, 64-row tiles in parts of unequal length. Within 1e-4 of every row's own
    maximum, the same bits from call to call, nothing written between the rows of C."""
    import gpu_util as gu
    import torch
    few = _weights(cr, kind, 61, k, seed=340 + m)
    cols = np.random.RandomState(m).randint(0, 61, n)
    a = synth.normal(341 + m, (m, k))
    ref = cr.gemm(cr.oracle(), kind, a, few, 61)[:, cols]
    w = capi.Weight(kind, n, k, np.ascontiguousarray(few.reshape(61, -1)[cols]))
    first = gu.gpu_matmul(w, a)
    dc = torch.full((m, n + 12), float("nan"), device="cuda")
    capi.matmul(w, gu.dev(a), m, dc, ldc=n + 12, stream=gu.stream())
    got = dc[:, :n].cpu().numpy()
    assert torch.isnan(dc[:, n:]).all(), "the call wrote between the rows of C"
    w.destroy()
    assert (np.abs(got - ref).max(axis=1) / np.abs(ref).max(axis=1)).max() <= gu.TOL
    assert np.array_equal(got, first), "the first call differs from the second"


@pytest.mark.parametrize("kind", ["q4_K", "q6_K"])
@pytest.mark.parametrize("m,n,k,off", [(33, 1001, 4096, 0), (96, 2502, 2304, 0), (130, 1503, 6400, 0), (40, 1000, 4096, 1)])
def test_k_format_gemm_in_parts_of_k_at_any_alignment(hipq, cr, kind, m, n, k, off):
    """Rows of one to three values behind the last quad, and an output that does not start on sixteen bytes: the product
    in parts has the bits of the one whose rows are padded to whole quads, and nothing is written beside its rows."""
    import gpu_util as gu
    import torch
    few = _weights(cr, kind, 61, k, seed=350 + m)
    pad = (n + 3) // 4 * 4
    cols = np.random.RandomState(n).randint(0, 61, pad)
    a = synth.normal(351 + m, (m, k))
    ref = cr.gemm(cr.oracle(), kind, a, few, 61)[:, cols[:n]]
    blocks = np.ascontiguousarray(few.reshape(61, -1)[cols])
    even, w = capi.Weight(kind, pad, k, blocks), capi.Weight(kind, n, k, np.ascontiguousarray(blocks[:n]))
    want = gu.gpu_matmul(even, a)[:, :n]
    buf = torch.full((m * n + off + 5,), float("nan"), device="cuda")
    capi.matmul(w, gu.dev(a), m, buf[off:off + m * n], stream=gu.stream())
    torch.cuda.synchronize()
    got = buf.cpu().numpy()
    assert np.isnan(got[:off]).all() and np.isnan(got[off + m * n:]).all(), "the call wrote beside C"
    got = got[off:off + m * n].reshape(m, n)
    for x in (even, w):
        x.destroy()
    assert np.array_equal(got, want)
    assert (np.abs(got - ref).max(axis=1) / np.abs(ref).max(axis=1)).max() <= gu.TOL


@pytest.mark.parametrize("kind", ["q4_K", "q6_K"])
@pytest.mark.parametrize("m", [17, 32, 33, 97, 130])
def test_k_format_gemm_of_32_row_tiles(hipq, cr, kind, m):
    """Tiles of 32 rows: every quarter of the quantizer's 128-row tiles, an odd number of super-blocks, columns past the last
    tile; one product, three weights in a launch and the gated pair."""
    import gpu_util as gu
    import torch
    k, ns = 768, (1100, 70, 33)
    blocks = [_weights(cr, kind, n, k, seed=360 + n) for n in ns]
    a = synth.normal(361 + m, (m, k))
    refs = [cr.gemm(cr.oracle(), kind, a, b, n) for b, n in zip(blocks, ns)]
    ws = [capi.Weight(kind, n, k, b) for b, n in zip(blocks, ns)]
    mul = capi.Weight(kind, ns[0], k, np.ascontiguousarray(blocks[0].reshape(ns[0], -1)[::-1]))
    try:
        outs = [torch.full((m, n), float("nan"), device="cuda") for n in ns]
        capi.matmul_multi(ws, gu.dev(a), m, outs, stream=gu.stream())
        h = torch.full((m, ns[0]), float("nan"), device="cuda")
        capi.mlp_swiglu(ws[0], mul, gu.dev(a), m, h, stream=gu.stream())
        torch.cuda.synchronize()
        for got, ref in [(gu.gpu_matmul(ws[0], a), refs[0])] + [(o.cpu().numpy(), r) for o, r in zip(outs, refs)]:
            assert not np.isnan(got).any()
            assert (np.abs(got - ref).max(axis=1) / np.abs(ref).max(axis=1)).max() <= gu.TOL
        assert gu.rel_err(h.cpu().numpy(), cr.swiglu(refs[0], refs[0][:, ::-1])) <= gu.TOL
    finally:
        for w in ws + [mul]:
            w.destroy()


@pytest.mark.parametrize("m,k", [(2, 256), (7, 1280), (17, 1024)])
def test_q4_K_rows_of_their_own_with_hard_super_blocks(hipq, cr, m, k):
    """The row form of the quantizer, sixteen values a lane: rounding adversaries, a row of zeros, a largest magnitude with both
    signs (the first decides), strided rows; a last wavefront that is not full. The reference's bits of every row alone."""
    import os
    import gpu_util as gu
    import torch
    adv = np.load(os.path.join(os.path.dirname(__file__), "golden", "q8k_rounding_adversaries.npy")).reshape(-1, 256)
    n = 1030
    blocks = _weights(cr, "q4_K", n, k, seed=380 + m)
    a = synth.normal(381 + m, (m, k))
    for r in range(m):
        a[r, (r % (k // 256)) * 256:][:256] = adv[r % len(adv)]
    a[1] = 0.0
    a[m - 1, 7], a[m - 1, 200], a[m - 1, 90] = 9.25, -9.25, -9.25
    ref = np.concatenate([cr.gemm(cr.oracle(), "q4_K", a[r:r + 1], blocks, n) for r in range(m)])
    w = capi.Weight("q4_K", n, k, blocks)
    wide = torch.full((m, k + 8), float("nan"), device="cuda")
    wide[:, :k] = gu.dev(a)
    out = torch.full((m, n), float("nan"), device="cuda")
    capi.matmul_each_row(w, wide, m, out, lda=k + 8, stream=gu.stream())
    torch.cuda.synchronize()
    w.destroy()
    assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.astype(np.float32).view(np.uint32))


@pytest.mark.parametrize("m,n,k", [(2, 20001, 256), (3, 12310, 512), (5, 9001, 1280), (8, 4100, 1024), (9, 1030, 2304), (16, 610, 256),
                                   (13, 4100, 4352)])
def test_q6_K_few_rows_on_the_matrix_cores(hipq, cr, m, n, k):
    """One pass and two of eight rows, a last pass of one row and more, one round of super-blocks, whole rounds and a part of
    one, columns behind the last tile of 32, strided rows: every row has the bits of its own product, as one call and as rows of
    their own, before and after the weight's tile copy exists."""
    import gpu_util as gu
    import torch
    few = _weights(cr, "q6_K", 61, k, seed=390 + m)
    cols = np.random.RandomState(n).randint(0, 61, n)
    a = synth.normal(391 + m, (m, k))
    a[m // 2] = 0.0
    ref = np.concatenate([cr.gemm(cr.oracle(), "q6_K", a[r:r + 1], few, 61) for r in range(m)])[:, cols].astype(np.float32)
    w = capi.Weight("q6_K", n, k, np.ascontiguousarray(few.reshape(61, -1)[cols]))
    wide = torch.full((m, k + 4), float("nan"), device="cuda")
    wide[:, :k] = gu.dev(a)
    try:
        for _ in range(2):
            out = torch.full((m, n + 5), float("nan"), device="cuda")
            capi.matmul_each_row(w, wide, m, out, lda=k + 4, ldc=n + 5, stream=gu.stream())
            torch.cuda.synchronize()
            got = out.cpu().numpy()
            assert np.isnan(got[:, n:]).all(), "the call wrote between the rows of C"
            assert np.array_equal(got[:, :n].copy().view(np.uint32), ref.view(np.uint32))
        one = gu.gpu_matmul(w, a)
    finally:
        w.destroy()
    if m <= (4 if n * k >= 2 ** 25 else 8 if n * k >= 2 ** 24 else 16):
        assert np.array_equal(one.view(np.uint32), ref.view(np.uint32))
    else:
        assert gu.rel_err(one, ref) <= gu.TOL


def test_q6_K_few_rows_captured_before_the_copy_exists(hipq, cr):
    """The few-rows Q6_K kernel reads a copy of the weight that its first product makes; a call that is being captured, and the
    one that may not allocate, use the weight as it is stored: the same bits, replayed three times with the copy made between."""
    import gpu_util as gu
    import torch
    m, n, k = 8, 5000, 512
    blocks = _weights(cr, "q6_K", n, k, seed=395)
    fresh, warm = capi.Weight("q6_K", n, k, blocks), capi.Weight("q6_K", n, k, blocks)
    a = gu.dev(synth.normal(396, (m, k)))
    want, out, na = (torch.full((m, n), float("nan"), device="cuda") for _ in range(3))
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        capi.matmul(warm, a, m, want, stream=side.cuda_stream)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        capi.matmul(fresh, a, m, out, stream=torch.cuda.current_stream().cuda_stream)
    capi.matmul_noalloc(fresh, a, m, na, stream=gu.stream())
    torch.cuda.synchronize()
    assert torch.equal(na, want)
    for _ in range(3):
        out.fill_(-1.0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        eager = torch.full((m, n), float("nan"), device="cuda")
        capi.matmul(fresh, a, m, eager, stream=gu.stream())
        torch.cuda.synchronize()
        assert torch.equal(eager, want)
    fresh.destroy(), warm.destroy()


@pytest.mark.parametrize("m,n,k", [(40, 8192, 512), (18, 12100, 1024), (24, 1100, 8192), (17, 87360, 256), (64, 2048, 4096)])
def test_q4_K_few_rows_or_tiles(hipq, cr, m, n, k):
    """Seventeen to 64 rows up to (column tiles) x (passes of eight rows) x (super-blocks) = 8192, where the interface promises
    the reference's bits whatever is the faster: one product, the first of two weights, and rows that are products of their
    own. The second weight of the call, too narrow for the promise, within 1e-4."""
    import gpu_util as gu
    import torch
    few = _weights(cr, "q4_K", 61, k, seed=370 + m)
    cols = np.random.RandomState(n).randint(0, 61, n)
    a = synth.normal(371 + m, (m, k))
    ref = cr.gemm(cr.oracle(), "q4_K", a, few, 61)[:, cols]
    alone = np.concatenate([cr.gemm(cr.oracle(), "q4_K", a[i:i + 1], few, 61) for i in range(m)])[:, cols]
    w = capi.Weight("q4_K", n, k, np.ascontiguousarray(few.reshape(61, -1)[cols]))
    v = capi.Weight("q4_K", 61, k, few)
    outs = [torch.full((m, x), float("nan"), device="cuda") for x in (n, 61, n)]
    capi.matmul_multi([w, v], gu.dev(a), m, outs[:2], stream=gu.stream())
    capi.matmul_each_row(w, gu.dev(a), m, outs[2], stream=gu.stream())
    torch.cuda.synchronize()
    got = [o.cpu().numpy() for o in outs] + [gu.gpu_matmul(w, a)]
    w.destroy(), v.destroy()
    for x in (got[0], got[3]):
        assert np.array_equal(x.view(np.uint32), ref.astype(np.float32).view(np.uint32))
    assert gu.rel_err(got[1], cr.gemm(cr.oracle(), "q4_K", a, few, 61)) <= gu.TOL
    assert np.array_equal(got[2].view(np.uint32), alone.astype(np.float32).view(np.uint32))


@pytest.mark.parametrize("m,k,ns", [(64, 1024, (6000, 6000)), (64, 2048, (2048, 2048, 2048)), (40, 512, (4100, 1030, 8000, 1024)),
                                    (33, 4096, (1536, 1024))])
def test_matmul_multi_q4_K_beyond_sixteen_rows_equals_the_single_calls(hipq, cr, m, k, ns):
    """Several Q4_K weights a call on both sides of what one launch of the few-rows kernel takes: every output has the bits
    of hipq_matmul against that weight, which are the reference's at these sizes; the gated pair of the first two agrees with
    the reference's products."""
    import gpu_util as gu
    import torch
    few = _weights(cr, "q4_K", 61, k, seed=390 + m)
    a = synth.normal(391 + m, (m, k))
    ref = cr.gemm(cr.oracle(), "q4_K", a, few, 61)
    cols = [np.random.RandomState(n + i).randint(0, 61, n) for i, n in enumerate(ns)]
    ws = [capi.Weight("q4_K", n, k, np.ascontiguousarray(few.reshape(61, -1)[c])) for n, c in zip(ns, cols)]
    try:
        outs = [torch.full((m, n), float("nan"), device="cuda") for n in ns]
        capi.matmul_multi(ws, gu.dev(a), m, outs, stream=gu.stream())
        torch.cuda.synchronize()
        for w, o, c in zip(ws, outs, cols):
            got = o.cpu().numpy().view(np.uint32)
            assert np.array_equal(got, gu.gpu_matmul(w, a).view(np.uint32)), w.n
            assert np.array_equal(got, ref[:, c].astype(np.float32).view(np.uint32)), w.n
        if ns[0] == ns[1]:
            h = torch.full((m, ns[0]), float("nan"), device="cuda")
            capi.mlp_swiglu(ws[0], ws[1], gu.dev(a), m, h, stream=gu.stream())
            torch.cuda.synchronize()
            assert gu.rel_err(h.cpu().numpy(), cr.swiglu(ref[:, cols[0]], ref[:, cols[1]])) <= gu.TOL
    finally:
        for w in ws:
            w.destroy()


def test_q4_K_gemm_tall_tiles(hipq, cr):
    """A shape for which the Q4_K GEMM picks its 128-row tiles (two rounds of 64-row
    tiles against one of 128-row tiles), with M not a multiple of the tile height."""
    import gpu_util as gu
    m, n, k = 1000, 8192, 512
    blocks = _weights(cr, "q4_K", n, k, seed=47)
    a = synth.normal(447, (m, k))
    ref = cr.gemm(cr.oracle(), "q4_K", a, blocks, n)
    w = capi.Weight("q4_K", n, k, blocks)
    got = gu.gpu_matmul(w, a)
    w.destroy()
    assert not np.isnan(got).any()
    assert gu.rel_err(got, ref) <= gu.TOL, gu.rel_err(got, ref)


@pytest.mark.parametrize("kind", ["q4_0", "q4_K"])
def test_x8_layout_equals_canonical(hipq, cr, kind):
    """Weights handed over in NNTrainer's 8-row interleave give the same outputs."""
    import gpu_util as gu
    n, k = 512, 1024
    blocks = _weights(cr, kind, n, k, seed=51)
    x8 = cr.repack_x8(cr.oracle(), kind, blocks, n, k)
    a = synth.normal(52, (5, k))
    w0 = capi.Weight(kind, n, k, blocks)
    w1 = capi.Weight(kind, n, k, x8, layout=capi.LAYOUT_X8)
    c0, c1 = gu.gpu_matmul(w0, a), gu.gpu_matmul(w1, a)
    w0.destroy(); w1.destroy()
    assert np.array_equal(c0, c1)


def test_host_memory_entry(hipq, cr):
    """HIPQ_MEM_HOST: plain host pointers in and out, with row strides."""
    import gpu_util as gu
    n, k, m = 256, 512, 3
    blocks = _weights(cr, "q4_K", n, k, seed=61)
    a = np.zeros((m, k + 64), np.float32)
    a[:, :k] = synth.normal(62, (m, k))
    c = np.full((m, n + 16), np.nan, np.float32)
    w = capi.Weight("q4_K", n, k, blocks)
    capi.matmul(w, a, m, c, lda=k + 64, ldc=n + 16, mem=capi.MEM_HOST)
    w.destroy()
    ref = cr.gemm(cr.oracle(), "q4_K", a[:, :k], blocks, n)
    assert gu.rel_err(c[:, :n], ref) <= gu.TOL
    assert np.isnan(c[:, n:]).all()


def test_matmul_multi_shares_quantization(hipq, cr):
    import gpu_util as gu
    import torch
    k, m = 1024, 1
    ns = [512, 256, 256]
    blocks = [_weights(cr, "q4_0", n, k, seed=70 + i) for i, n in enumerate(ns)]
    ws = [capi.Weight("q4_0", n, k, b) for n, b in zip(ns, blocks)]
    a = synth.normal(73, (m, k))
    da = gu.dev(a)
    outs = [torch.empty((m, n), device="cuda") for n in ns]
    capi.matmul_multi(ws, da, m, outs, stream=gu.stream())
    torch.cuda.synchronize()
    for n, b, o in zip(ns, blocks, outs):
        assert gu.rel_err(o.cpu().numpy(), cr.gemm(cr.oracle(), "q4_0", a, b, n)) <= gu.TOL
    for w in ws:
        w.destroy()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,k", [(8, 256), (37, 256), (1000, 768), (1024, 1024), (3072, 1024), (2050, 2048),
                                 (4096, 4096), (8200, 3072), (12288, 4096)])
def test_decode_row_quantized_in_the_gemv_equals_the_two_launches(hipq, cr, kind, n, k):
    """hipq_matmul with one row on a small matrix runs one kernel whose workgroups
    quantize the row themselves; the multi-weight entry with more than four weights
    keeps the quantizer kernel and the GEMV on its blocks. Same arithmetic, so the
    outputs are the same bits; the oracle pins both."""
    import gpu_util as gu
    import torch
    blocks = _weights(cr, kind, n, k, seed=500 + n)
    a = synth.normal(600 + k, (1, k))
    a[0, 5] = 0.0
    if k >= 512:
        a[0, 256:512] = 0.0   # an all-zero block: scale 0
    w = capi.Weight(kind, n, k, blocks)
    one = gu.gpu_matmul(w, a)
    two = [torch.full((1, n), float("nan"), device="cuda") for _ in range(5)]
    capi.matmul_multi([w] * 5, gu.dev(a), 1, two, stream=gu.stream())
    torch.cuda.synchronize()
    w.destroy()
    for t in two:
        assert np.array_equal(one, t.cpu().numpy())
    ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
    assert gu.rel_err(one, ref) <= gu.TOL


@pytest.mark.parametrize("kind,k", [("q4_0", 32), ("q4_0", 96), ("q4_0", 1024), ("q4_0", 2048), ("q4_0", 2080),
                                    ("q4_0", 4096), ("q4_K", 256), ("q4_K", 2304), ("q4_K", 4096), ("q6_K", 256),
                                    ("q6_K", 4096)])
def test_decode_row_of_unusual_values_is_quantized_like_the_reference(hipq, cr, kind, k):
    """The quantization inside the decode GEMV: blocks of zeros, of one value, of tiny and of large values, and
    largest magnitudes that occur with both signs (the K-formats' scale takes the first one's). Same bits."""
    import gpu_util as gu
    n = 200
    blocks = _weights(cr, kind, n, k, seed=2000 + k)
    w = capi.Weight(kind, n, k, blocks)
    blk = 32 if kind == "q4_0" else 256
    for case in range(6):
        a = synth.normal(2001 + k + case, (1, k)).reshape(-1, blk)
        top = np.abs(a).max() * 1.5
        for i in range(a.shape[0]):
            lo, hi = (7 * i + 5 * case) % 16, 16 + (11 * i + 3 * case) % (blk - 16)
            if case == 0:
                a[i, lo], a[i, hi] = top, -top
            elif case == 1:
                a[i, lo], a[i, hi] = -top, top
            elif case == 2 and i % 2 == 0:
                a[i] = 0.0
            elif case == 3:
                a[i] *= 1e-37 if i % 3 else 1e30
            elif case == 4:
                a[i] = a[i, 0]
            elif case == 5:
                a[i, lo], a[i, lo ^ 1] = top, -top
        a = a.reshape(1, k)
        ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
        got = gu.gpu_matmul(w, a)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (case, got[0, :4], ref[0, :4])
    w.destroy()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("k,ns", [(1024, [2048, 1024, 1024]), (1024, [3072, 3072]), (256, [8, 37, 4, 130]),
                                  (4096, [4096]), (2048, [1000, 6150])])
def test_decode_row_on_several_weights_is_one_launch_with_the_same_bits(hipq, cr, kind, k, ns):
    """Up to four weights of one format and K on one row go out as a single launch
    (Q, K and V, or gate and up, of a decoder layer); the outputs are those of
    hipq_matmul on each weight."""
    import gpu_util as gu
    import torch
    blocks = [_weights(cr, kind, n, k, seed=700 + n + i) for i, n in enumerate(ns)]
    ws = [capi.Weight(kind, n, k, b) for n, b in zip(ns, blocks)]
    a = synth.normal(710 + k, (1, k))
    outs = [torch.full((1, n), float("nan"), device="cuda") for n in ns]
    capi.matmul_multi(ws, gu.dev(a), 1, outs, stream=gu.stream())
    torch.cuda.synchronize()
    for w, b, n, o in zip(ws, blocks, ns, outs):
        assert np.array_equal(o.cpu().numpy(), gu.gpu_matmul(w, a))
        assert gu.rel_err(o.cpu().numpy(), cr.gemm(cr.oracle(), kind, a, b, n)) <= gu.TOL
    for w in ws:
        w.destroy()


def test_decode_calls_replay_from_a_captured_graph(hipq, cr):
    """The one-row calls are single kernel launches without allocations, so a caller
    can capture a decoder layer's FCs in a graph. Every replay, with other work on
    the device in between, gives the bits of the direct calls."""
    import gpu_util as gu
    import torch
    k, ns = 1024, [2048, 1024, 1024]
    blocks = [_weights(cr, "q4_0", n, k, seed=800 + i) for i, n in enumerate(ns)]
    ws = [capi.Weight("q4_0", n, k, b) for n, b in zip(ns, blocks)]
    wo = capi.Weight("q4_0", k, 2048, _weights(cr, "q4_0", k, 2048, seed=810))
    x = torch.zeros((1, k), device="cuda")
    qkv = [torch.zeros((1, n), device="cuda") for n in ns]
    y = torch.zeros((1, k), device="cuda")

    def layer(stream):
        capi.matmul_multi(ws, x, 1, qkv, stream=stream)
        capi.matmul(wo, qkv[0], 1, y, stream=stream)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        layer(side.cuda_stream)          # first calls outside the capture
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        layer(side.cuda_stream)
    for it in range(4):
        x.copy_(gu.dev(synth.normal(820 + it, (1, k))))
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in qkv] + [y.clone()]
        scratch = torch.randn(1 << 20, device="cuda").sum()   # other work between the replays
        layer(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        for g, e in zip(got, qkv + [y]):
            assert torch.equal(g, e), "replay %d differs from the direct calls" % it
        assert torch.isfinite(scratch)
    for w in ws + [wo]:
        w.destroy()


@pytest.mark.parametrize("own_streams", [False, True])
def test_calls_from_several_threads(hipq, cr, own_streams):
    """The entry points are called from several threads (the reference's expert loop
    runs Tensor::dot inside an OpenMP loop, qwen_moe_layer.cpp:478-490; model load uses a
    thread per node). Calls that name the same stream share its scratch: their launches
    must not interleave. Every result equals the one a single thread gets."""
    import threading
    import gpu_util as gu
    import torch
    n, k = 384, 512
    ws = {kind: capi.Weight(kind, n, k, _weights(cr, kind, n, k, seed=950)) for kind in ("q4_0", "q4_K")}
    cases = [(kind, m) for kind in ws for m in (1, 5, 40)]
    acts = {m: gu.dev(synth.normal(960 + m, (m, k))) for m in (1, 5, 40)}
    want = {}
    for kind, m in cases:
        c = torch.empty((m, n), device="cuda")
        capi.matmul(ws[kind], acts[m], m, c, stream=gu.stream())
        torch.cuda.synchronize()
        want[(kind, m)] = c.clone()
    errors = []

    def work(tid):
        try:
            st = torch.cuda.Stream() if own_streams else torch.cuda.current_stream()
            outs = {cs: torch.empty((cs[1], n), device="cuda") for cs in cases}
            for it in range(25):
                for kind, m in cases[tid % 2:] + cases[:tid % 2]:
                    capi.matmul(ws[kind], acts[m], m, outs[(kind, m)], stream=st.cuda_stream)
                st.synchronize()
                for cs in cases:
                    if not torch.equal(outs[cs], want[cs]):
                        errors.append((tid, it, cs))
                        return
        except Exception as e:  # noqa: BLE001 - reported below
            errors.append((tid, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for w in ws.values():
        w.destroy()
    assert not errors, errors[:3]


def test_weights_read_from_a_model_file(hipq, cr, tmp_path):
    """A file laid out as NNTrainer writes MODEL_FORMAT_BIN (tensors back to back, Q4_0 and
    Q4_K in the 8-row interleave, a scheme word in front of Q4_K only): the handles read
    from it multiply like handles made from the same bytes."""
    import gpu_util as gu
    specs = [("q4_0", 512, 1024), ("q4_K", 256, 512), ("q6_K", 384, 256), ("q4_K", 128, 256)]
    blocks = [_weights(cr, kind, n, k, seed=900 + i) for i, (kind, n, k) in enumerate(specs)]
    stored = [cr.repack_x8(cr.oracle(), kind, b, n, k) if kind != "q6_K" else b
              for (kind, n, k), b in zip(specs, blocks)]
    path = tmp_path / "model.bin"
    listing = [("skip", 4096)]
    with open(path, "wb") as f:
        f.write(b"\0" * 7)                            # the caller's start offset
        f.write(np.arange(1024, dtype=np.float32).tobytes())
        for (kind, n, k), b in zip(specs, stored):
            if kind == "q4_K":
                f.write(np.uint16(3).tobytes())       # QScheme::Q4_Kx8
            f.write(np.ascontiguousarray(b).tobytes())
            listing.append((kind, n, k, capi.LAYOUT_X8 if kind != "q6_K" else capi.LAYOUT_CANONICAL))
        f.write(b"tail")
    ws, end = capi.weights_from_file(path, listing, offset=7)
    assert ws[0] is None and end == path.stat().st_size - 4
    for w, (kind, n, k), b in zip(ws[1:], specs, blocks):
        a = synth.normal(910 + n, (3, k))
        ref = capi.Weight(kind, n, k, b)
        assert np.array_equal(gu.gpu_matmul(w, a), gu.gpu_matmul(ref, a))
        ref.destroy()
        w.destroy()
    # a Q4_Kx8 tensor listed as canonical, and a file that ends early, leave no handle behind
    with pytest.raises(capi.HipqError):
        capi.weights_from_file(path, [("skip", 4096), ("q4_0", 512, 1024, capi.LAYOUT_X8), ("q4_K", 256, 512)],
                               offset=7)
    with pytest.raises(capi.HipqError):
        capi.weights_from_file(path, listing + [("q6_K", 4096, 4096)], offset=7)


@pytest.mark.parametrize("kind,m", [("q4_K", 1), ("q4_K", 40), ("q6_K", 3), ("q6_K", 40)])
def test_matmul_multi_other_formats_and_prefill(hipq, cr, kind, m):
    """The multi-weight entry with the Q8_K formats, one row and a prefill chunk (the
    Q4_K prefill goes through the tiled activations and the matrix-core GEMM)."""
    import gpu_util as gu
    import torch
    k = 512
    ns = [384, 128, 256]
    blocks = [_weights(cr, kind, n, k, seed=80 + i) for i, n in enumerate(ns)]
    ws = [capi.Weight(kind, n, k, b) for n, b in zip(ns, blocks)]
    a = synth.normal(83, (m, k))
    outs = [torch.full((m, n), float("nan"), device="cuda") for n in ns]
    capi.matmul_multi(ws, gu.dev(a), m, outs, stream=gu.stream())
    torch.cuda.synchronize()
    for n, b, o in zip(ns, blocks, outs):
        got = o.cpu().numpy()
        assert not np.isnan(got).any()
        assert gu.rel_err(got, cr.gemm(cr.oracle(), kind, a, b, n)) <= gu.TOL
    for w in ws:
        w.destroy()


@pytest.mark.parametrize("m", [4, 6])
def test_matmul_multi_few_rows_mixed_paths(hipq, cr, m):
    """A few rows against Q4_K weights of different sizes (and a Q6_K one) in one multi-weight call:
    the large Q4_K matrices take the matrix-core kernel (one quantization in its row form shared by
    them), the small one and the Q6_K one the GEMV engine with their own quantizations. All carry
    the reference's bits, whatever the order of the weights in the call."""
    import gpu_util as gu
    import torch
    k = 1024
    kinds, ns = ["q4_K", "q4_K", "q6_K", "q4_K", "q4_K"], [8192, 512, 640, 1056, 8200]
    blocks = [_weights(cr, kd, n, k, seed=95 + i) for i, (kd, n) in enumerate(zip(kinds, ns))]
    ws = [capi.Weight(kd, n, k, b) for kd, n, b in zip(kinds, ns, blocks)]
    a = synth.normal(99 + m, (m, k))
    outs = [torch.full((m, n), float("nan"), device="cuda") for n in ns]
    capi.matmul_multi(ws, gu.dev(a), m, outs, stream=gu.stream())
    torch.cuda.synchronize()
    for kd, n, b, o in zip(kinds, ns, blocks, outs):
        ref = cr.gemm(cr.oracle(), kd, a, b, n)
        assert np.array_equal(o.cpu().numpy().view(np.uint32), ref.view(np.uint32)), (kd, n)
    for w in ws:
        w.destroy()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("k", [4096, 3072, 2304, 1024])
def test_matmul_multi_one_row_one_launch_by_row_length(hipq, cr, kind, k):
    """One row against the Q, K, V of a layer (one launch that quantizes the row itself): the launch with the
    row length as a constant (4096, 3072, 1024) and for any length (2304), widths that end inside a
    wavefront's group of rows. Every output carries the reference's bits."""
    import gpu_util as gu
    import torch
    ns = [4100, 1024, 1030] if k >= 3072 else [2050, 520, 512]
    blocks = [_weights(cr, kind, n, k, seed=1450 + i) for i, n in enumerate(ns)]
    ws = [capi.Weight(kind, n, k, b) for n, b in zip(ns, blocks)]
    a = synth.normal(1460 + k % 13, (1, k))
    outs = [torch.full((1, n), float("nan"), device="cuda") for n in ns]
    capi.matmul_multi(ws, gu.dev(a), 1, outs, stream=gu.stream())
    torch.cuda.synchronize()
    for n, b, o in zip(ns, blocks, outs):
        got = o.cpu().numpy()
        ref = cr.gemm(cr.oracle(), kind, a, b, n)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (n, gu.rel_err(got, ref))
    for w in ws:
        w.destroy()


@pytest.mark.parametrize("m,k", [(2, 1024), (8, 1280), (13, 256), (16, 2048), (40, 1024), (64, 512)])
def test_matmul_multi_q4_0_few_rows_one_launch(hipq, cr, m, k):
    """A few rows against several Q4_0 weights of one K (Q, K, V or gate, up of a decode step of a
    batch): the weights' column tiles side by side in one launch of the few-rows kernel, four
    weights a launch (five make a launch of four and a single product), widths that end inside a
    32-column tile, outputs with a row stride. Every output carries the reference's bits."""
    import gpu_util as gu
    import torch
    ns = [2048, 1000, 1024, 72, 520]
    blocks = [_weights(cr, "q4_0", n, k, seed=1400 + i) for i, n in enumerate(ns)]
    ws = [capi.Weight("q4_0", n, k, b) for n, b in zip(ns, blocks)]
    a = synth.normal(1410 + m, (m, k))
    outs = [torch.full((m, n + 8 * i), float("nan"), device="cuda") for i, n in enumerate(ns)]
    capi.matmul_multi(ws, gu.dev(a), m, outs, ldc=[n + 8 * i for i, n in enumerate(ns)], stream=gu.stream())
    torch.cuda.synchronize()
    for i, (n, b, o) in enumerate(zip(ns, blocks, outs)):
        got = o.cpu().numpy()
        ref = cr.gemm(cr.oracle(), "q4_0", a, b, n)
        assert np.array_equal(got[:, :n].view(np.uint32), ref.view(np.uint32)), (n, gu.rel_err(got[:, :n], ref))
        assert np.isnan(got[:, n:]).all(), "the call wrote between the rows of an output"
    for w in ws:
        w.destroy()


@pytest.mark.parametrize("m,k", [(2, 1024), (3, 512), (6, 1280), (13, 256), (16, 2048), (40, 1024)])
def test_matmul_multi_q4_K_few_rows_one_launch(hipq, cr, m, k):
    """The same for Q4_K weights: one quantization in the row form of the matrix-core kernels (rows
    below 4 * (m / 4) under the 4-row rule), then the weights' column tiles side by side in one launch
    of gemm_rows_q4k.hip, four weights a launch. The reference's bits for every output, and the bits
    of the single-weight call where that one keeps them (the single call of a wide weight with more
    than 16 rows takes the prefill GEMM, which agrees to 1e-4)."""
    import gpu_util as gu
    import torch
    ns = [2048, 1000, 1024, 72, 520]
    blocks = [_weights(cr, "q4_K", n, k, seed=1500 + i) for i, n in enumerate(ns)]
    ws = [capi.Weight("q4_K", n, k, b) for n, b in zip(ns, blocks)]
    a = synth.normal(1510 + m, (m, k))
    a[1, 3] = 8.5
    a[1, 7] = -8.5
    outs = [torch.full((m, n + 8 * i), float("nan"), device="cuda") for i, n in enumerate(ns)]
    capi.matmul_multi(ws, gu.dev(a), m, outs, ldc=[n + 8 * i for i, n in enumerate(ns)], stream=gu.stream())
    torch.cuda.synchronize()
    for i, (n, b, o) in enumerate(zip(ns, blocks, outs)):
        got = o.cpu().numpy()
        ref = cr.gemm(cr.oracle(), "q4_K", a, b, n)
        assert np.array_equal(got[:, :n].view(np.uint32), ref.view(np.uint32)), (n, gu.rel_err(got[:, :n], ref))
        assert np.isnan(got[:, n:]).all(), "the call wrote between the rows of an output"
    for w in ws:
        w.destroy()


@pytest.mark.parametrize("ns", [[72, 3072], [3072, 72, 1000]])
def test_matmul_multi_q6_K_members_of_different_size_share_the_quantization(hipq, cr, ns):
    """Q6_K weights of one multi-weight call share the quantized rows of the first one's product. A
    product of few tiles keeps its partial products of parts of K behind those rows in the same
    workspace, and a later, larger member needs more of it: the workspace is sized for the largest
    member before the first product, so that it does not move between them. A fresh stream, so that
    the workspace starts empty."""
    import gpu_util as gu
    import torch
    m, k = 65, 2048
    blocks = [_weights(cr, "q6_K", n, k, seed=1700 + i) for i, n in enumerate(ns)]
    ws = [capi.Weight("q6_K", n, k, b) for n, b in zip(ns, blocks)]
    a = synth.normal(1710, (m, k))
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        da = gu.dev(a)
        outs = [torch.full((m, n), float("nan"), device="cuda") for n in ns]
        side.synchronize()
        capi.matmul_multi(ws, da, m, outs, stream=side.cuda_stream)
        side.synchronize()
    for n, b, o in zip(ns, blocks, outs):
        got = o.cpu().numpy()
        assert not np.isnan(got).any()
        assert gu.rel_err(got, cr.gemm(cr.oracle(), "q6_K", a, b, n)) <= gu.TOL, n
    for w in ws:
        w.destroy()


def test_matmul_multi_seeded_mixed_calls(hipq, cr):
    """Forty multi-weight calls drawn from a seeded generator: one to seven weights of mixed formats
    and widths, one to 130 rows, every second call on a stream of its own (an empty workspace).
    Whatever grouping the call chooses (one launch for several weights, shared quantizations, parts
    of K), every output is within 1e-4 of the reference and Q4_0 outputs carry its bits."""
    import gpu_util as gu
    import torch
    rng = np.random.default_rng(7)
    cache = {}

    def blocks_of(kind, n, k):
        if (kind, n, k) not in cache:
            cache[(kind, n, k)] = _weights(cr, kind, n, k, seed=2000 + n + k + len(kind))
        return cache[(kind, n, k)]

    for it in range(40):
        k = int(rng.choice([256, 512, 1024, 1280, 2048]))
        cnt = int(rng.integers(1, 8))
        kinds = [str(rng.choice(["q4_0", "q4_0", "q4_K", "q4_K", "q6_K"])) for _ in range(cnt)]
        ns = [int(rng.choice([72, 256, 520, 1000, 1024, 2048, 3072, 4100])) for _ in range(cnt)]
        m = int(rng.choice([1, 2, 3, 4, 5, 8, 9, 13, 16, 17, 31, 40, 64, 65, 130]))
        a = synth.normal(3000 + it, (m, k))
        if m > 1:
            a[1, 3] = 7.5
            a[1, 9] = -7.5
        blocks = [blocks_of(kd, n, k) for kd, n in zip(kinds, ns)]
        ws = [capi.Weight(kd, n, k, b) for kd, n, b in zip(kinds, ns, blocks)]
        outs = [torch.full((m, n), float("nan"), device="cuda") for n in ns]
        da = gu.dev(a)
        st = torch.cuda.Stream() if it % 2 else torch.cuda.current_stream()
        torch.cuda.synchronize()
        capi.matmul_multi(ws, da, m, outs, stream=st.cuda_stream)
        torch.cuda.synchronize()
        for kd, n, b, o in zip(kinds, ns, blocks, outs):
            got = o.cpu().numpy()
            ref = cr.gemm(cr.oracle(), kd, a, b, n)
            case = (it, m, k, kd, n)
            assert not np.isnan(got).any(), case
            assert gu.rel_err(got, ref) <= gu.TOL, case
            if kd == "q4_0":
                assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), case
        for w in ws:
            w.destroy()


def test_matmul_multi_mixed_k_formats_prefill(hipq, cr):
    """Q4_K and Q6_K weights in one multi-weight prefill call: both take tiled Q8_K activations, but
    the reference quantizes the rows of a Q4_K product four at a time and those of a Q6_K product one
    by one (different sign rules), so the two groups must not share one quantization. Row 2 holds
    +amax before -amax, where the two quantizers differ."""
    import gpu_util as gu
    import torch
    m, k = 40, 512
    kinds, ns = ["q4_K", "q6_K", "q4_K", "q6_K"], [256, 160, 128, 384]
    blocks = [_weights(cr, kd, n, k, seed=90 + i) for i, (kd, n) in enumerate(zip(kinds, ns))]
    ws = [capi.Weight(kd, n, k, b) for kd, n, b in zip(kinds, ns, blocks)]
    a = synth.normal(93, (m, k))
    a[2, 5] = 9.5
    a[2, 9] = -9.5
    outs = [torch.full((m, n), float("nan"), device="cuda") for n in ns]
    capi.matmul_multi(ws, gu.dev(a), m, outs, stream=gu.stream())
    torch.cuda.synchronize()
    for kd, n, b, o, w in zip(kinds, ns, blocks, outs, ws):
        got = o.cpu().numpy()
        assert not np.isnan(got).any()
        assert gu.rel_err(got, cr.gemm(cr.oracle(), kd, a, b, n)) <= gu.TOL
        assert np.array_equal(got, gu.gpu_matmul(w, a)), "the multi-weight call differs from the single one"
    for w in ws:
        w.destroy()


@pytest.mark.parametrize("kind", ["q4_K", "q4_0"])
def test_matmul_multi_prefill_five_weights_one_launch_per_four(hipq, cr, kind):
    """Prefill products of several weights go out up to four a launch (column tiles of the weights
    side by side in one grid): five weights make a launch of four and one of one; widths that are
    no multiple of the workgroup's column tile; every output equals the single-weight call's."""
    import gpu_util as gu
    import torch
    m, k = 300, 1024
    ns = [512, 96, 200, 1024, 136]
    blocks = [_weights(cr, kind, n, k, seed=110 + i) for i, n in enumerate(ns)]
    ws = [capi.Weight(kind, n, k, b) for n, b in zip(ns, blocks)]
    a = synth.normal(113, (m, k))
    outs = [torch.full((m, n), float("nan"), device="cuda") for n in ns]
    capi.matmul_multi(ws, gu.dev(a), m, outs, stream=gu.stream())
    torch.cuda.synchronize()
    for n, b, o, w in zip(ns, blocks, outs, ws):
        got = o.cpu().numpy()
        assert not np.isnan(got).any()
        assert gu.rel_err(got, cr.gemm(cr.oracle(), kind, a, b, n)) <= gu.TOL
        assert np.array_equal(got, gu.gpu_matmul(w, a)), "the multi-weight call differs from the single one"
    for w in ws:
        w.destroy()


def test_bad_arguments_are_reported(hipq):
    with pytest.raises(capi.HipqError) as e:
        capi.weight_nbytes("q4_K", 16, 100)  # K not a multiple of 256 (q4_k_tensor.cpp:23-27)
    assert e.value.code == -1
    blocks = np.zeros(capi.weight_nbytes("q6_K", 8, 256), np.uint8)
    with pytest.raises(capi.HipqError):
        capi.Weight("q6_K", 8, 256, blocks, layout=capi.LAYOUT_X8)  # no x8 form of Q6_K
    blocks = np.zeros(capi.weight_nbytes("q4_0", 12, 64), np.uint8)
    with pytest.raises(capi.HipqError):
        capi.Weight("q4_0", 12, 64, blocks, layout=capi.LAYOUT_X8)  # N % 8 != 0 (repack returns -1)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows,n,k", [(8, 1100, 1024), (5, 512, 768), (12, 2048, 512), (16, 300, 256),
                                      (37, 1056, 1024), (3, 8200, 512), (1, 640, 256), (70, 1030, 512)])
def test_matmul_each_row_has_the_bits_of_single_row_products(hipq, cr, kind, rows, n, k):
    """hipq_matmul_each_row: the rows of a batch of decode steps against one weight in one call, every
    row with the bits of its own M = 1 product (the reference's loop over batch entries). For Q4_K
    that differs from hipq_matmul with M = rows (no 4-row quantizer, no pairwise sums): row 1 holds
    +amax before -amax, where the two quantizers round differently. Large and small matrices (the
    matrix-core kernel and the GEMV engine), more than 16 rows (several steps), strided rows, and
    host memory."""
    import gpu_util as gu
    import torch
    blocks = _weights(cr, kind, n, k, seed=500 + n)
    a = synth.normal(501 + rows + k, (rows, k))
    if rows > 1:
        a[1, 3] = 7.25
        a[1, 11] = -7.25
    ref = np.concatenate([cr.gemm(cr.oracle(), kind, a[r:r + 1], blocks, n) for r in range(rows)], axis=0)
    w = capi.Weight(kind, n, k, blocks)
    try:
        lda, ldc = k + 64, n + 32
        da = torch.zeros((rows, lda), device="cuda")
        da[:, :k] = gu.dev(a)
        dc = torch.full((rows, ldc), float("nan"), device="cuda")
        capi.matmul_each_row(w, da, rows, dc, lda=lda, ldc=ldc, stream=gu.stream())
        torch.cuda.synchronize()
        got = dc[:, :n].cpu().numpy()
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), \
            "%d of %d outputs differ in bits" % ((got.view(np.uint32) != ref.view(np.uint32)).sum(), got.size)
        assert torch.isnan(dc[:, n:]).all(), "the call wrote between the rows of C"
        host = np.full((rows, n), np.nan, np.float32)
        capi.matmul_each_row(w, a, rows, host, mem=capi.MEM_HOST, stream=gu.stream())
        assert np.array_equal(host.view(np.uint32), ref.view(np.uint32))
        single = gu.gpu_matmul(w, a[1:2]) if rows > 1 else None
        if single is not None:
            assert np.array_equal(single.view(np.uint32), ref[1:2].view(np.uint32))
    finally:
        w.destroy()


@pytest.mark.parametrize("rows,n,k", [(5, 1030, 256), (8, 1056, 2304), (13, 1100, 4352), (61, 1027, 1280), (16, 2049, 1024)])
def test_q4_K_few_rows_of_their_own_by_rounds(hipq, cr, rows, n, k):
    """Rows that are products of their own take the few-rows kernel whose records are super-block totals: one super-block, whole
    rounds of four and a rest of one, row counts that leave the last pass partly empty, columns beyond the last tile of 32.
    The bits of the row products."""
    import gpu_util as gu
    few = _weights(cr, "q4_K", 37, k, seed=2600 + k % 97)
    cols = np.random.RandomState(n).randint(0, 37, n)
    a = synth.normal(2601 + k % 89, (rows, k))
    ref = np.concatenate([cr.gemm(cr.oracle(), "q4_K", a[r:r + 1], few, 37) for r in range(rows)])[:, cols]
    w = capi.Weight("q4_K", n, k, np.ascontiguousarray(few.reshape(37, -1)[cols]))
    out = gu.dev(np.full((rows, n), np.nan, np.float32))
    capi.matmul_each_row(w, gu.dev(a), rows, out, stream=gu.stream())
    got = out.cpu().numpy()
    w.destroy()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


def test_row_counts_across_the_kernel_choices(hipq, cr):
    """hipq_matmul picks among the GEMV engine, the few-rows matrix-core kernel (one to eight passes),
    the prefill GEMMs (whole K or parts of K) by format, row count and matrix size. Shapes drawn
    around the thresholds from a seeded generator: every result within 1e-4 of the reference, Q4_0
    and every product of one or two rows with its bits, a second call the bits of the first."""
    import gpu_util as gu
    rng = np.random.RandomState(20250117)
    done = 0
    while done < 36:
        kind = KINDS[done % 3]
        n = int(rng.choice([1000, 1024, 1056, 2048, 4096, 4100, 8192, 8200]))
        k = int(rng.choice([256, 1024, 2048, 2304, 4096]))
        m = int(rng.choice([1, 2, 3, 4, 5, 8, 9, 12, 16, 17, 24, 33, 48, 64, 65, 70]))
        if m * n * k > 4e8:
            continue
        blocks = _weights(cr, kind, n, k, seed=1200 + done)
        a = synth.normal(1300 + done, (m, k))
        ref = cr.gemm(cr.oracle(), kind, a, blocks, n)
        w = capi.Weight(kind, n, k, blocks)
        got = gu.gpu_matmul(w, a)
        again = gu.gpu_matmul(w, a)
        w.destroy()
        case = (kind, m, n, k)
        assert not np.isnan(got).any(), case
        assert gu.rel_err(got, ref) <= gu.TOL, (case, gu.rel_err(got, ref))
        assert np.array_equal(got, again), case
        if kind == "q4_0" or m <= 2:
            assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), case
        done += 1



def _extreme_rows(m, k):
    """Rows whose Q8_0 block scales are infinite, subnormal and zero as fp16, in whole rows and in single blocks."""
    a = synth.normal(77, (m, k))
    for r in range(m):
        b = slice(32 * (r % (k // 32)), 32 * (r % (k // 32)) + 32)
        kind = r % 8
        if kind == 1:
            a[r] *= 3e7          # every scale infinite
        elif kind == 2:
            a[r, b] *= 1e9       # one infinite scale in the row
        elif kind == 3:
            a[r, b] = 0.0
            a[r, b.start] = -2e7  # one product of the block
        elif kind == 4:
            a[r] *= 1e-3         # subnormal scales
        elif kind == 5:
            a[r, b] *= 3e-6      # the smallest ones
        elif kind == 6:
            a[r] *= 1e-9         # scales of zero
        elif kind == 7:
            a[r, b] *= 65504 * 127 / np.abs(a[r, b]).max()  # the largest finite scale
    return a


@pytest.mark.parametrize("m,n,k", [(70, 130, 256), (97, 300, 1056), (2100, 520, 288)])
@pytest.mark.parametrize("call", ["matmul", "swiglu"])
def test_q4_0_on_six_bit_operands_with_extreme_scales(hipq, cr, call, m, n, k):
    """gemm_f6.hip: block scales that are infinite, subnormal and zero as fp16. An infinite scale makes the sums of its own
    row infinite (or NaN, where the reference's are), and no other block's: the reference's bits. Infinite and NaN
    activations give what the kernels that read the weight as stored give."""
    import gpu_util as gu
    import torch
    blocks = _weights(cr, "q4_0", n, k, seed=3000 + m)
    blocks2 = _weights(cr, "q4_0", n, k, seed=3001 + m)
    w, w2 = capi.Weight("q4_0", n, k, blocks), capi.Weight("q4_0", n, k, blocks2)

    def product(a):
        da, out = gu.dev(a), torch.full((m, n), 7.0, device="cuda")
        if call == "matmul":
            capi.matmul(w, da, m, out, stream=gu.stream())
        else:
            capi.mlp_swiglu(w, w2, da, m, out, stream=gu.stream())
        torch.cuda.synchronize()
        return out.cpu().numpy()

    def same(got, ref):
        nan = np.isnan(ref)
        assert np.array_equal(np.isnan(got), nan)
        bits = got.view(np.uint32) != ref.view(np.uint32)
        assert not (bits & ~nan).any(), "%d of %d outputs differ in bits" % ((bits & ~nan).sum(), got.size)

    a = _extreme_rows(m, k)
    if call == "matmul":
        ref = cr.gemm(cr.oracle(), "q4_0", a, blocks, n)
        assert np.isinf(ref).any() and np.isfinite(ref[2]).sum() == 0
        same(product(a), ref)
    # the stored weights' kernels, by a call that may not allocate
    v, v2 = capi.Weight("q4_0", n, k, blocks), capi.Weight("q4_0", n, k, blocks2)
    for extra in (0.0, np.inf, -np.inf, np.nan):
        if extra != 0.0:
            a[::5, 7] = extra
        da, y, z = gu.dev(a), torch.empty((m, n), device="cuda"), torch.empty((m, n), device="cuda")
        capi.matmul_noalloc(v, da, m, y, stream=gu.stream())
        capi.matmul_noalloc(v2, da, m, z, stream=gu.stream())
        torch.cuda.synchronize()
        y, z = y.cpu().numpy(), z.cpu().numpy()
        if call == "matmul":
            same(product(a), y)
        else:
            got = product(a)
            with np.errstate(all="ignore"):
                want = y / (1.0 + np.exp(-y.astype(np.float64))) * z
            assert np.array_equal(np.isnan(got), np.isnan(want))
            fine = np.isfinite(want)
            assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
            assert np.allclose(got[fine], want[fine], rtol=1e-5, atol=1e-30)
    for x in (w, w2, v, v2):
        x.destroy()
