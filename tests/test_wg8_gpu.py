"""The eight-wave tiled kernel (5_amd/csrc/hcg_wg8.h) at the edges of its tiles.

Small-integer operands make every sum exact in float32 whatever its order, so
C must equal A @ B bit for bit.  A and B are views into NaN-filled buffers
(NaN past K in A's rows and past N in B's: no element outside a view may reach
C) and C is a view into a NaN-filled buffer whose other elements must stay.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DEV = "cuda:0"
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}


def _padded(x, dtype, pad):
    rows, cols = x.shape
    buf = torch.full((rows + 1, cols + pad), float("nan"), dtype=dtype, device=DEV)
    buf[:rows, :cols] = torch.from_numpy(x.astype(np.float32)).to(DEV).to(dtype)
    return buf[:rows, :cols]


def _check(m, n, k, dtype, pad, algo="auto"):
    import hc.gfx950 as g

    print(f"case wg8 {dtype} m={m} n={n} k={k} pad={pad} algo={algo}", flush=True)
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    ai, bi = rng.integers(-4, 5, size=(m, k)), rng.integers(-4, 5, size=(k, n))
    a, b = _padded(ai, DTYPES[dtype], pad), _padded(bi, DTYPES[dtype], pad)
    guard = torch.full((m + 2, n + pad), float("nan"), dtype=torch.float32, device=DEV)
    for _ in range(2):  # the second call reuses the stream's workspace
        g.gemm(a, b, out=guard[:m, :n], algo=algo)
    torch.cuda.synchronize()
    got = guard.cpu().numpy()
    assert np.array_equal(got[:m, :n], (ai.astype(np.float64) @ bi.astype(np.float64)).astype(np.float32))
    assert np.all(np.isnan(got[m:])) and np.all(np.isnan(got[:, n:]))


# Tiles of 64x64 (one and two a side, K below, at and past one and several
# 64-wide steps), 64x128, 128x128 and 128x256, each with ragged and whole
# edges, as the plan picks them for these sizes.
_SHAPES = [
    (65, 65, 1), (65, 66, 63), (127, 129, 64), (129, 190, 257), (128, 128, 128), (500, 1000, 512),
    (200, 8192, 1000), (170, 6019, 264),
    (1664, 2000, 200), (1601, 2041, 264), (2048, 2048, 520),
    (2500, 2500, 1000), (576, 7232, 768), (8192, 1024, 1024),
]


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("m,n,k", _SHAPES)
def test_wg8_tiles(m, n, k, dtype):
    _check(m, n, k, dtype, 8)


@pytest.mark.parametrize("pad", [0, 1, 4, 5])
@pytest.mark.parametrize("m,n,k", [(129, 190, 261), (170, 6019, 70), (1601, 2041, 65)])
def test_wg8_row_alignment(m, n, k, pad):
    """Rows of A, B and C at every alignment class (K and N odd or not)."""
    _check(m, n, k, "float16", pad)


@pytest.mark.parametrize("m,n,k", [(512, 512, 16384), (130, 200, 8200), (128, 8192, 8192), (333, 444, 4999),
                                   (192, 136, 1536)])
def test_wg8_split_k(m, n, k):
    _check(m, n, k, "bfloat16", 4)
    _check(m, n, k, "float16", 3)


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (128, 128, 31), (129, 257, 96), (640, 384, 1000)])
def test_forced_128x128(m, n, k):
    _check(m, n, k, "float16", 4, "tiled_128x128")


# A transposed operand is read where it lies; the padding of its stored rows
# (past M for A stored K x M, past K for B stored N x K) holds NaN.
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("which", ["a", "b"])
@pytest.mark.parametrize("m,n,k", [(65, 65, 2), (130, 100, 63), (127, 129, 64), (129, 190, 257), (200, 8192, 1000),
                                   (1601, 2041, 264), (2500, 2500, 1001), (4095, 3001, 100), (4096, 4096, 72),
                                   (512, 512, 4104), (333, 444, 4999)])
@pytest.mark.parametrize("pad", [0, 3, 8])
def test_transposed_operand_in_place(m, n, k, which, dtype, pad):
    import hc.gfx950 as g

    print(f"case transposed {which} {dtype} m={m} n={n} k={k} pad={pad}", flush=True)
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    ai, bi = rng.integers(-4, 5, size=(m, k)), rng.integers(-4, 5, size=(k, n))
    a = _padded(ai.T, DTYPES[dtype], pad).t() if which == "a" else _padded(ai, DTYPES[dtype], pad)
    b = _padded(bi.T, DTYPES[dtype], pad).t() if which == "b" else _padded(bi, DTYPES[dtype], pad)
    guard = torch.full((m + 2, n + 5), float("nan"), dtype=torch.float32, device=DEV)
    g.gemm(a, b, out=guard[:m, :n])
    torch.cuda.synchronize()
    got = guard.cpu().numpy()
    want = (ai.astype(np.float64) @ bi.astype(np.float64)).astype(np.float32)
    assert np.array_equal(got[:m, :n], want)
    assert np.all(np.isnan(got[m:])) and np.all(np.isnan(got[:, n:]))
    assert torch.equal(g.gemm(a, b), torch.from_numpy(want).to(DEV))  # without out=


@pytest.mark.parametrize("m,n,k", [(64, 200, 96), (200, 64, 96), (3, 70, 8), (70, 70, 1), (100, 100, 40)])
def test_transposed_operands_the_kernel_declines_are_copied(m, n, k):
    """Few rows or columns, K = 1, and both operands transposed take the
    row-major path on copies."""
    import hc.gfx950 as g

    rng = np.random.default_rng(m + n + k)
    ai, bi = rng.integers(-4, 5, size=(m, k)), rng.integers(-4, 5, size=(k, n))
    a, b = _padded(ai, torch.float16, 1), _padded(bi, torch.float16, 1)
    at, bt = _padded(ai.T, torch.float16, 1).t(), _padded(bi.T, torch.float16, 1).t()
    want = torch.from_numpy((ai.astype(np.float64) @ bi.astype(np.float64)).astype(np.float32)).to(DEV)
    for x, y in ((at, bt), (at, b), (a, bt)):
        assert torch.equal(g.gemm(x, y), want)


def test_transposed_operand_under_capture():
    """A split-K call on a transposed operand replays from a graph, with eager
    calls between the replays, and repeats bit for bit."""
    import hc.gfx950 as g

    x = torch.randn(8192, 300, device=DEV).half()
    dy = torch.randn(8192, 200, device=DEV).half()
    out = torch.empty(300, 200, device=DEV)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        g.gemm(x.t(), dy, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        g.gemm(x.t(), dy, out=out)
    for _ in range(4):
        x.copy_(torch.randn_like(x))
        eager = g.gemm(x.t(), dy)
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


def _kernels_of(fn):
    """Names of the kernels a call runs."""
    from torch.profiler import ProfilerActivity, profile

    fn()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return [e.name for e in prof.events() if e.device_type == torch.autograd.DeviceType.CUDA]


# Over 1.25 row blocks of 64 per CU the narrow kernel walks several blocks per
# workgroup: a block's last stage beside the next one's first, K of one stage
# (so that every stage ends a block), below one and ragged, the last block
# ragged, workgroups with one block more than others.  33 to 64 columns of at
# most 64 MiB go to the tiled kernel unless the narrow one is asked for.
@pytest.mark.parametrize("m,n,k,algo", [(20481, 8, 128, "auto"), (20417, 1, 1, "auto"), (33000, 16, 130, "auto"),
                                        (40963, 17, 500, "auto"), (24000, 33, 1001, "narrow"),
                                        (32768, 64, 640, "narrow"), (50001, 40, 257, "narrow"),
                                        (20417, 50, 64, "narrow"), (40001, 40, 1001, "auto"),
                                        (20500, 64, 4096, "auto")])
@pytest.mark.parametrize("dtype", list(DTYPES))
def test_narrow_kernel_walks_row_blocks(m, n, k, algo, dtype):
    import hc.gfx950 as g

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the line is 1.25 row blocks per CU, stated here for 256")
    _check(m, n, k, dtype, 3 if dtype == "float16" else 8, algo)
    a = torch.zeros(m, k, dtype=DTYPES[dtype], device=DEV)
    b = torch.zeros(k, n, dtype=DTYPES[dtype], device=DEV)
    out = torch.empty(m, n, device=DEV)
    names = _kernels_of(lambda: g.gemm(a, b, out=out, algo=algo))
    block = 16 if n <= 16 else 32 if n <= 32 else 64
    walking = f"gemm_rowstream_kernel<{list(DTYPES).index(dtype)}, {block}, false, 0, true>"
    assert any(walking in name for name in names), names


# K splits summed by a block's last workgroup against the same partials summed
# by a second launch, which hcg_gemm_noalloc keeps: in the same order, so bit
# for bit, with new operands every round (a stale partial would show).  The
# streaming kernel with one, two and four row blocks at their most splits, N
# ragged or not; the narrow kernel with 16, 32 and 64 columns; and one split
# more than each takes, where both calls run the second launch.
@pytest.mark.parametrize("m,n,k,kernel,summed", [
    (16, 8191, 8192, "stream", True), (1, 1001, 2050, "stream", True), (16, 1000, 2560, "stream", False),
    (31, 5001, 5000, "stream", True), (31, 4099, 5000, "stream", False),
    (40, 9001, 8191, "stream", True), (64, 8192, 8200, "stream", False),
    (4096, 13, 8192, "rowstream", True), (200, 12, 8192, "rowstream", True), (300, 5, 900, "rowstream", True),
    (2048, 24, 12000, "rowstream", True), (400, 24, 5120, "rowstream", False),
    (2048, 57, 12001, "rowstream", True), (1000, 33, 12001, "rowstream", False)])
def test_summed_splits_match_the_reduce_launch(m, n, k, kernel, summed):
    import hc.gfx950 as g
    from hc.gfx950 import _native

    print(f"case summed splits m={m} n={n} k={k}", flush=True)
    lib = _native.load()
    stream = torch.cuda.current_stream().cuda_stream
    for rnd in range(4):
        gen = torch.Generator(device=DEV).manual_seed(rnd)
        a = torch.randn((m, k), generator=gen, device=DEV).half()
        b = torch.randn((k, n), generator=gen, device=DEV).half()
        outs = []
        for entry in (lib.hcg_gemm, lib.hcg_gemm_noalloc):
            c = torch.full((m, n), float("nan"), dtype=torch.float32, device=DEV)
            rc = entry(_native.HCG_F16, a.data_ptr(), k, b.data_ptr(), n, c.data_ptr(), n, m, n, k, stream)
            assert rc == _native.HCG_OK, _native.last_error(lib)
            outs.append(c)
        torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[1]), rnd
    names = _kernels_of(lambda: g.gemm(a, b, out=outs[0]))
    assert any(f"gemm_{kernel}_kernel" in name for name in names), names
    assert any("reduce" in name for name in names) == (not summed), names


# 17 to 64 rows and 33 to 64 columns: small operands take the tiled kernel,
# larger ones and long K stream; both sides of each line.
@pytest.mark.parametrize("m,n,k", [(16, 300, 500), (17, 65, 500), (32, 300, 4096), (32, 300, 4097),
                                   (33, 300, 8192), (33, 300, 8193), (33, 1000, 999),
                                   (64, 8192, 4096), (64, 8200, 4096), (64, 4001, 8191), (500, 32, 500),
                                   (500, 33, 500), (17, 33, 100), (16, 33, 100), (4096, 64, 8192), (4104, 64, 8192),
                                   (64, 64, 8200), (3001, 57, 777)])
@pytest.mark.parametrize("pad", [0, 8])
def test_few_rows_or_columns_either_route(m, n, k, pad):
    _check(m, n, k, "float16", pad)


# Operands within the size rules above whose rows lie so far apart that they
# span 2 GiB or more stream as before: the tiled kernel's small tiles and K
# splits are for 32-bit offsets.  The same kernel gives the same bits.
@pytest.mark.parametrize("m,n,k,lda,ldb,algo", [
    (32, 512, 4096, 4096, 300000, "skinny"), (33, 520, 8000, 8000, 140001, "skinny"),
    (64, 300, 4096, 4096, 262144, "skinny"), (4096, 64, 1000, 300000, 64, "narrow"),
    (3000, 40, 513, 400001, 40, "narrow")])
def test_few_rows_or_columns_of_a_wide_matrix_stream(m, n, k, lda, ldb, algo):
    import hc.gfx950 as g

    print(f"case wide rows m={m} n={n} k={k} lda={lda} ldb={ldb}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(m + n + k)
    a = torch.full((m, lda), float("nan"), dtype=torch.float16, device=DEV)[:, :k]
    b = torch.full((k, ldb), float("nan"), dtype=torch.float16, device=DEV)[:, :n]
    a.copy_(torch.randn(a.shape, generator=gen, device=DEV))
    b.copy_(torch.randn(b.shape, generator=gen, device=DEV))
    got = g.gemm(a, b)
    assert torch.equal(got, g.gemm(a, b, algo=algo))
    want = a.double() @ b.double()
    # 32-bit sums of k exact products, in any order: each within k units of 2^-24 of the sum of magnitudes.
    assert ((got - want).abs() <= k * 2.0**-24 * (a.double().abs() @ b.double().abs())).all()


# Rows so far apart that an operand spans 2 GiB: the WIDE form of
# gemm_dma_kernel, whose 128x128 tiles are the fastest while the larger ones
# leave CUs idle.
@pytest.mark.parametrize("m,n,k,lda,tile", [(4097, 128, 512, 300000, "128, 128"), (4096, 1000, 40, 300000, "128, 128"),
                                            (16000, 1000, 64, 80000, "128, 256"),
                                            (4096, 4096, 1024, 300000, "256, 256")])
def test_wide_tiles_by_size(m, n, k, lda, tile):
    import hc.gfx950 as g

    print(f"case wide tiles m={m} n={n} k={k} lda={lda}", flush=True)
    rng = np.random.default_rng(m + n + k)
    ai, bi = rng.integers(-4, 5, size=(m, k)), rng.integers(-4, 5, size=(k, n))
    a = torch.full((m, lda), float("nan"), dtype=torch.float16, device=DEV)[:, :k]
    a.copy_(torch.from_numpy(ai.astype(np.float32)))
    b = torch.from_numpy(bi.astype(np.float32)).to(DEV).half()
    out = torch.empty(m, n, device=DEV)
    names = _kernels_of(lambda: g.gemm(a, b, out=out))
    assert np.array_equal(out.cpu().numpy(), (ai.astype(np.float64) @ bi.astype(np.float64)).astype(np.float32))
    assert any(f"gemm_dma_kernel<0, {tile}, " in name for name in names), names


# K splits whose partials an eager call sums in its last workgroups (tiled,
# transposed, streaming, narrow): captured, a second launch sums them, in the
# same order and with nothing to clear.
@pytest.mark.parametrize("m,n,k,which", [(512, 512, 16384, ""), (103, 254, 779, ""), (300, 200, 8192, "a"),
                                         (300, 200, 8192, "b"), (16, 4096, 4096, ""), (31, 4099, 5000, ""),
                                         (2048, 24, 12000, ""), (300, 5, 900, "")])
def test_captured_splits_match_eager_and_clear_nothing(m, n, k, which):
    import hc.gfx950 as g

    print(f"case captured splits m={m} n={n} k={k} {which}", flush=True)
    x = torch.empty((k, m) if which == "a" else (m, k), dtype=torch.float16, device=DEV)
    y = torch.empty((n, k) if which == "b" else (k, n), dtype=torch.float16, device=DEV)
    a, b = x.t() if which == "a" else x, y.t() if which == "b" else y
    out, eager = torch.empty(m, n, device=DEV), torch.empty(m, n, device=DEV)
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        g.gemm(a, b, out=eager)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        for _ in range(2):  # back to back: the second's partials overwrite the first's
            g.gemm(a, b, out=out)
    names = _kernels_of(graph.replay)
    assert any("gemm" in name for name in names) and not any("fill_zero" in name for name in names), names
    for seed in range(4):
        gen = torch.Generator(device=DEV).manual_seed(seed)
        x.copy_(torch.randn(x.shape, generator=gen, device=DEV))
        y.copy_(torch.randn(y.shape, generator=gen, device=DEV))
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            g.gemm(a, b, out=eager)
        torch.cuda.synchronize()
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), seed


# Under many rows a transposed B is copied to row-major first (both sides of the
# line at three K; A stored transposed never is).
@pytest.mark.parametrize("m,n,k,copied", [(64000, 66, 1024, False), (64300, 66, 1024, True), (32900, 65, 4096, False),
                                          (33200, 65, 4096, True), (11200, 100, 16400, False),
                                          (11300, 100, 16400, True)])
def test_transposed_b_under_many_rows_is_copied(m, n, k, copied):
    import hc.gfx950 as g
    from hc.gfx950 import _native

    print(f"case transposed b under many rows m={m} n={n} k={k}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(m + k)
    a = torch.randint(-3, 4, (m, k), generator=gen, device=DEV).half()
    bt = torch.randint(-3, 4, (n, k), generator=gen, device=DEV).half()
    c = torch.full((m, n), float("nan"), device=DEV)
    lib = _native.load()
    rc = lib.hcg_gemm_trans(_native.HCG_F16, 0, a.data_ptr(), k, 1, bt.data_ptr(), k, c.data_ptr(), n, m, n, k,
                            torch.cuda.current_stream().cuda_stream or None)
    assert rc == (_native.HCG_EDECLINED if copied else _native.HCG_OK), _native.last_error(lib)
    got = g.gemm(a, bt.t())
    want = torch.empty_like(c)  # |sums| < 2^24: exact in float32 in any order
    for i in range(0, m, 8192):
        want[i : i + 8192] = a[i : i + 8192].float() @ bt.t().float().contiguous()
    assert torch.equal(got, want)
    assert torch.isnan(c).all() if copied else torch.equal(c, want)
    at = a[:8200].t().contiguous().t()
    assert torch.equal(g.gemm(at, bt.t().contiguous()), want[:8200])


# Past one 64-column tile per CU, 17 to 32 rows with K up to N / 32 and 33 to 64
# with K up to 128 stream.
@pytest.mark.parametrize("m,n,k,kernel", [(17, 16384, 96, "wg8"), (17, 16385, 96, "stream"), (32, 16640, 520, "stream"),
                                          (32, 16640, 521, "wg8"), (33, 16400, 128, "stream"),
                                          (64, 16400, 129, "wg8")])
def test_short_k_past_one_tile_per_cu_streams(m, n, k, kernel):
    import hc.gfx950 as g

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the line is one 64-column tile per CU, stated here for 256")
    _check(m, n, k, "float16", 8)
    a = torch.zeros(m, k, dtype=torch.float16, device=DEV)
    b = torch.zeros(k, n, dtype=torch.float16, device=DEV)
    out = torch.empty(m, n, device=DEV)
    names = _kernels_of(lambda: g.gemm(a, b, out=out))
    assert any(f"gemm_{kernel}_kernel" in name for name in names), names


# A remainder past a multiple of 256 is peeled onto a streaming kernel only for
# a gain the model can tell.
@pytest.mark.parametrize("m,n,k,peeled", [(4209, 3984, 552, False), (5440, 2848, 513, False), (4100, 4096, 768, True)])
def test_remainders_are_peeled_for_a_clear_gain(m, n, k, peeled):
    import hc.gfx950 as g

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the model's gains are stated here for 256 CUs")
    _check(m, n, k, "float16", 8)
    a = torch.zeros(m, k, dtype=torch.float16, device=DEV)
    b = torch.zeros(k, n, dtype=torch.float16, device=DEV)
    out = torch.empty(m, n, device=DEV)
    names = _kernels_of(lambda: g.gemm(a, b, out=out))
    assert any("gemm_dma_kernel" in name for name in names)
    assert any("gemm_stream_kernel" in name or "gemm_rowstream_kernel" in name for name in names) == peeled, names
