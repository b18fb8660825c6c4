"""GPU parity of the projections either side of the core (qwen35/kernels.py:291-319 fused_gemv, qwen35/batch.py:295-301
rms_rows) against the numpy restatement.  rms_rows is bit exact.  The product accumulates 1024 .. 3584 bf16 x bf16 terms in
float32 on the matrix cores (the reference accumulates them in float32 in another order, the restatement in float64), so its
bf16 outputs may differ by one rounding step: the tolerance is 1 bf16 ulp (2 after the add / swiglu epilogues, which round a
second time) plus 2e-5 of the largest output for sums that nearly cancel, and 2e-3 relative in the l2 norm."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import gdn_oracle as O
from tests.util import *  # noqa: F401,F403

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def qt():
    import qwen_tailor_amd as q
    q._lib.lib()
    return q


@pytest.mark.parametrize("M,K", [(1, 1024), (5, 1024), (64, 1024), (64, 2048), (3, 3584), (67, 520), (2, 8)])
def test_rms_rows_bit_exact(qt, dev, M, K):
    g = torch.Generator().manual_seed(M * 131 + K)
    x = rand_bf(g, (M, K), 1.7)
    nw = bf(1.0 + 0.2 * torch.randn(K, generator=g).numpy())
    got = qt.batch.rms_rows(to_dev(x, dev, BF16), to_dev(nw, dev, BF16), 1e-6)
    check_equal("rms_rows", to_np(got), O.rms_rows(x, nw, 1e-6))
    wide = qt.batch.rms_rows(to_dev(x, dev, BF16), to_dev(nw, dev, BF16), 1e-6, f32=True)
    assert wide.dtype == torch.float32 and torch.equal(wide, got.float())


def _close(name, got, want, ulps, inner=None):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    # the rounding step of the larger binade, plus an absolute term for sums that nearly cancel (float32 accumulation of K terms)
    tol = ulps * ulp_bf16(np.maximum(np.abs(got), np.abs(want))) + 2e-5 * np.abs(want).max()
    if inner is not None:        # an epilogue that rounds the product first: one rounding step of that (possibly larger) value
        tol = tol + ulp_bf16(np.abs(np.asarray(inner, np.float64)))
    bad = np.abs(got - want) > tol
    assert not bad.any(), f"{name}: {int(bad.sum())} of {bad.size} outputs beyond {ulps} bf16 ulp, worst {np.abs(got - want).max():.3g}"
    assert rel_l2(got, want) < 2e-3, f"{name}: rel l2 {rel_l2(got, want):.3g}"


# the six projections of a layer at decode time (hidden 1024, inter 3584), ragged row counts, a narrow and an odd-sized output
@pytest.mark.parametrize("M,N,K,epi", [
    (64, 8224, 1024, "none"), (64, 1024, 2048, "add"), (64, 5120, 1024, "none"), (64, 7168, 1024, "swiglu"), (64, 1024, 3584, "add"),
    (1, 8224, 1024, "none"), (5, 1024, 2048, "add"), (16, 7168, 1024, "swiglu"), (37, 264, 512, "none"), (70, 40, 512, "add"),
    (130, 1024, 1024, "none"), (3, 50, 512, "swiglu"),
    # wide outputs with K = 1024: rows in LDS from 4 to 64 rows (every count of 16-row blocks, partial blocks, feature counts
    # that leave the last workgroup partly or wholly past N); more than 64 rows keep the rows in registers
    (4, 8224, 1024, "none"), (17, 4096, 1024, "add"), (33, 7168, 1024, "swiglu"), (48, 4100, 1024, "none"), (63, 5120, 1024, "add"),
    (100, 8224, 1024, "none"), (3, 8224, 1024, "none"),
    # ... with each epilogue, and more row blocks than one pass of 64 rows
    (100, 4096, 1024, "add"), (70, 7168, 1024, "swiglu"), (200, 5120, 1024, "none")])
def test_fused_gemv_vs_oracle(qt, dev, M, N, K, epi):
    g = torch.Generator().manual_seed(M * 7 + N * 3 + K)
    W = rand_bf(g, (N, K), K ** -0.5)
    x = rand_bf(g, (M, K), 1.0)
    res = rand_bf(g, (M, N), 1.0) if epi == "add" else None
    got = qt.kernels.fused_gemv(to_dev(W, dev, BF16), to_dev(x, dev, BF16), res=None if res is None else to_dev(res, dev, BF16),
                                swiglu=epi == "swiglu")
    want = O.fused_gemv(W, x, res=res, swiglu=epi == "swiglu")
    assert tuple(got.shape) == want.shape
    # add: y = BF(BF(s) + res); when s and res nearly cancel, a product that rounds the other way moves y by one step of s
    _close(f"fused_gemv {epi}", to_np(got), want, 1 if epi == "none" else 2,
           inner=np.asarray(want, np.float64) - np.asarray(res, np.float64) if epi == "add" else None)


def test_fused_gemv_exact_on_small_integers(qt, dev):
    """with small-integer data every partial sum is exact in float32, whatever the order: the product must match bit for bit"""
    g = torch.Generator().manual_seed(11)
    M, N, K = 33, 96, 1024
    W = torch.randint(-3, 4, (N, K), generator=g).float().numpy()
    x = torch.randint(-2, 3, (M, K), generator=g).float().numpy()
    got = qt.kernels.fused_gemv(to_dev(W, dev, BF16), to_dev(x, dev, BF16))
    check_equal("integer product", to_np(got), O.fused_gemv(W, x))


@pytest.mark.parametrize("M,N,epi", [(33, 4112, 0), (64, 8224, 1), (16, 4096, 2), (5, 5120, 0)])
def test_wide_projection_exact_and_any_output_alignment(qt, dev, M, N, epi):
    """The kernel for wide outputs at K = 1024 (rows in LDS) on small-integer data, where every order of summation gives the
    same bits; and the same call through the C ABI with y and res 2 bytes off an 8-byte boundary (the general kernels take
    over) must give the same bits."""
    from qwen_tailor_amd import _lib as QL
    g = torch.Generator().manual_seed(M + N + epi)
    K = 1024
    W = torch.randint(-3, 4, (N, K), generator=g).float().numpy()
    x = torch.randint(-2, 3, (M, K), generator=g).float().numpy()
    res = torch.randint(-9, 10, (M, N), generator=g).float().numpy() if epi == 1 else None
    dW, dx = to_dev(W, dev, BF16), to_dev(x, dev, BF16)
    dres = None if res is None else to_dev(res, dev, BF16)
    got = qt.kernels.fused_gemv(dW, dx, res=dres, swiglu=epi == 2)
    want = O.fused_gemv(W, x, res=res, swiglu=epi == 2)
    if epi == 2:
        _close("integer swiglu", to_np(got), want, 1)            # silu of an integer is not an integer: within one rounding
    else:
        check_equal("integer product", to_np(got), want)
    NO = N // 2 if epi == 2 else N
    ybuf = torch.zeros(M * NO + 8, dtype=BF16, device=dev)
    rbuf = torch.zeros(M * N + 8, dtype=BF16, device=dev)
    if dres is not None:
        rbuf[1:1 + M * N] = dres.reshape(-1)
    QL.call("qt_fused_gemv", QL.ptr(dW), QL.ptr(dx), ctypes.c_void_p(rbuf.data_ptr() + 2) if dres is not None else None,
            ctypes.c_void_p(ybuf.data_ptr() + 2), M, N, K, epi, QL.stream())
    assert torch.equal(ybuf[1:1 + M * NO].reshape(M, NO), got), "outputs off an 8-byte boundary differ"


# edges of the row blocks (16, 32, 48, 64, 96, 128 rows) and of the feature tiles (32 or 64 features; 8224 = 514 blocks of 16, more
# than two per CU by two; 4100 = a last block of 4 features; 5132 = 64 x 80 + 12)
@pytest.mark.parametrize("M,N,epi", [
    (1, 4096, 0), (1, 8224, 2), (15, 4100, 0), (16, 8224, 1), (17, 5132, 0), (32, 8224, 2), (33, 4100, 1), (48, 8224, 0), (49, 8224, 1),
    (64, 5132, 2), (65, 4100, 0), (80, 8224, 1), (96, 7168, 2), (97, 8224, 0), (128, 5132, 1), (129, 4096, 0), (257, 4100, 2)])
def test_wide_projection_tiles_and_fused_rms_prologue(qt, dev, M, N, epi):
    _check_wide(qt, dev, M, N, epi)


# the last N of a tile that leaves a workgroup per CU and the first beyond it (256 CUs x 32 or 64 features + one more block for a
# sixteenth of the CUs), by rows; beyond it the rms prologue is a launch of its own from 17 rows on
@pytest.mark.parametrize("M,N,epi", [
    (16, 8452, 0), (17, 8448, 0), (17, 8452, 1), (32, 16384, 2), (32, 16640, 0), (32, 16644, 1), (33, 8448, 2), (48, 8452, 0), (40, 16640, 1),
    (48, 16644, 2), (49, 8320, 0), (64, 8324, 2), (50, 16644, 1), (65, 5520, 0), (96, 5524, 2), (96, 8320, 1), (66, 8324, 0)])
def test_wide_projection_beyond_a_workgroup_per_cu(qt, dev, M, N, epi):
    _check_wide(qt, dev, M, N, epi)


def _check_wide(qt, dev, M, N, epi):
    """exact on small integers (every order of summation gives the same bits); with the rms prologue, in one launch up to 96 rows,
    the bits of the two calls"""
    g = torch.Generator().manual_seed(M * 5 + N + epi)
    K = 1024
    W = to_dev(torch.randint(-3, 4, (N, K), generator=g).float().numpy(), dev, BF16)
    x = torch.randint(-2, 3, (M, K), generator=g).float().numpy()
    res = torch.randint(-9, 10, (M, N), generator=g).float().numpy() if epi == 1 else None
    dres = None if res is None else to_dev(res, dev, BF16)
    got = qt.kernels.fused_gemv(W, to_dev(x, dev, BF16), res=dres, swiglu=epi == 2)
    want = O.fused_gemv(to_np(W), x, res=res, swiglu=epi == 2)
    if epi == 2:
        _close("integer swiglu", to_np(got), want, 1)
    else:
        check_equal("integer product", to_np(got), want)
    r = to_dev(rand_bf(g, (M, K), 1.3), dev, BF16)
    nw = to_dev(bf(1.0 + 0.2 * torch.randn(K, generator=g).numpy()), dev, BF16)
    one = qt.kernels.fused_gemv(W, r, nw=nw, res=dres, swiglu=epi == 2)
    two = qt.kernels.fused_gemv(W, qt.kernels.rms_rows(r, nw), res=dres, swiglu=epi == 2)
    assert torch.equal(one, two), "rms prologue in the launch and on its own differ"


# a few features more than whole tiles: one group of four, several, the most that the first tiles take; one and two row groups, 32 and 64
# features a tile
@pytest.mark.parametrize("M,N,epi", [(1, 8196, 0), (7, 8204, 2), (16, 8448, 1), (30, 8196, 1), (45, 8220, 0), (64, 8196, 2), (64, 8320, 1), (16, 8444, 2)])
def test_wide_projection_with_a_few_features_more(qt, dev, M, N, epi):
    _check_wide(qt, dev, M, N, epi)


# edges of the 4 x 4, 8 x 8, 8 x 16 and 16 x 16 tiles, outputs and rows that end inside a tile, K shorter than one batch of every
# wavefront (256, 512), not a multiple of the wavefronts' steps (1280, 3584) and longer than one batch (4352)
@pytest.mark.parametrize("M,N,K,epi", [
    (1, 1024, 2048, 1), (1, 50, 256, 2), (3, 1027, 1280, 0), (4, 2048, 3584, 1), (5, 1024, 3584, 1), (8, 4090, 2048, 2), (9, 1030, 2048, 0),
    (16, 1024, 4352, 1), (17, 1024, 2048, 1), (31, 1021, 3584, 0), (33, 1000, 2048, 2), (64, 1024, 3584, 1), (63, 1023, 3584, 0),
    (64, 1024, 2048, 1), (5, 16, 512, 0), (40, 40, 256, 1), (65, 1024, 3584, 1), (96, 1026, 2048, 2), (81, 1000, 512, 0), (128, 1020, 1280, 1),
    (97, 1024, 2048, 0), (30, 3070, 4352, 1)])
def test_narrow_projection_tiles_exact_on_small_integers(qt, dev, M, N, K, epi):
    g = torch.Generator().manual_seed(M * 3 + N + K + epi)
    W = torch.randint(-3, 4, (N, K), generator=g).float().numpy()
    x = torch.randint(-2, 3, (M, K), generator=g).float().numpy()
    res = torch.randint(-9, 10, (M, N), generator=g).float().numpy() if epi == 1 else None
    got = qt.kernels.fused_gemv(to_dev(W, dev, BF16), to_dev(x, dev, BF16), res=None if res is None else to_dev(res, dev, BF16), swiglu=epi == 2)
    want = O.fused_gemv(W, x, res=res, swiglu=epi == 2)
    if epi == 2:
        _close("integer swiglu", to_np(got), want, 1)
    else:
        check_equal("integer product", to_np(got), want)


# 16 x 16 tiles through LDS (one per CU where 8 x 16 would take two): outputs and rows that end inside a tile, wavefronts with one and with two
# steps of K (1280: two of ten wavefronts' steps; 1792), the fewest and the most tiles of the rule
@pytest.mark.parametrize("M,N,K", [(33, 1024, 2048), (64, 1023, 2048), (48, 1030, 1280), (96, 520, 1792), (17, 2047, 1536), (32, 2034, 2048), (9, 4095, 1280), (16, 4096, 2048),
                                   (130, 260, 2048), (257, 130, 1280)])
def test_narrow_projection_one_tile_per_cu(qt, dev, M, N, K):
    """exact on small integers, and on real values the bits of the same rows in batches of up to 16 (which smaller tiles take)"""
    cus, wgs = torch.cuda.get_device_properties(dev).multi_processor_count, lambda f: ((N + f - 1) // f) * ((M + 15) // 16)
    assert M > 8 and 1024 < K <= 2048 and wgs(16) <= cus < wgs(8), "not a case of this kernel"
    for epi in (0, 1) + ((2,) if N % 2 == 0 else ()):
        test_narrow_projection_tiles_exact_on_small_integers(qt, dev, M, N, K, epi)
    g = torch.Generator().manual_seed(M + N + K)
    W, x = (torch.randn((N, K), generator=g) * K ** -0.5).to(BF16).to(dev), torch.randn((M, K), generator=g).to(BF16).to(dev)
    few = 16 if N <= 1024 else 8 if N <= 2050 else 4
    check_tensors_equal("rows", qt.kernels.fused_gemv(W, x), torch.cat([qt.kernels.fused_gemv(W, x[i:i + few]) for i in range(0, M, few)]))


# K of one trip (up to 1024): every wavefront with two steps, with one, with one of two, and none for some
@pytest.mark.parametrize("K", [1024, 512, 768, 256])
@pytest.mark.parametrize("M,N", [(1, 2048), (3, 1027), (17, 2050), (80, 520)])
def test_narrow_projection_of_one_trip(qt, dev, M, N, K):
    for epi in (0, 1) + ((2,) if N % 2 == 0 else ()):
        test_narrow_projection_tiles_exact_on_small_integers(qt, dev, M, N, K, epi)


def test_the_residual_costs_a_narrow_projection_nothing(qt, dev):
    """it is requested behind the operands: 0.987 - 0.998 of the time without it (1.057 - 1.074 when it stood ahead of them; the bound
    lies between)"""
    g = torch.Generator().manual_seed(5)
    W, x, res = (to_dev(rand_bf(g, s, 0.03), dev, BF16) for s in ((2048, 768), (4, 768), (4, 2048)))
    without, with_res = graph_us(lambda: qt.kernels.fused_gemv(W, x)), graph_us(lambda: qt.kernels.fused_gemv(W, x, res=res))
    assert with_res < 1.03 * without, (with_res, without)


def test_fused_gemv_prologues_and_leading_dims(qt, dev):
    """nw = rms_rows first; gnorm = gated norm first (same bits as the stand-alone kernels, qwen35/batch.py:241-248);
    leading dimensions are flattened and restored; float32 x holding bf16 values is taken as is"""
    g = torch.Generator().manual_seed(12)
    W = to_dev(rand_bf(g, (256, 1024), 0.03), dev, BF16)
    x = to_dev(rand_bf(g, (2, 3, 1024), 1.0), dev, BF16)
    nw = to_dev(bf(1.0 + 0.1 * torch.randn(1024, generator=g).numpy()), dev, BF16)
    a = qt.kernels.fused_gemv(W, x, nw=nw)
    b = qt.kernels.fused_gemv(W, qt.batch.rms_rows(x.reshape(6, 1024), nw, f32=True))
    assert tuple(a.shape) == (2, 3, 256) and torch.equal(a.reshape(6, 256), b)
    Wo = to_dev(rand_bf(g, (128, 2048), 0.02), dev, BF16)
    y = to_dev(rand_bf(g, (4, 2048), 1.0), dev, BF16)
    proj = to_dev(rand_bf(g, (4, PW), 1.0), dev, BF16)
    gw = to_dev((1.0 + 0.1 * torch.randn(128, generator=g)).numpy().astype(np.float32), dev)
    res = to_dev(rand_bf(g, (4, 128), 1.0), dev, BF16)
    c = qt.kernels.fused_gemv(Wo, y, gnorm=(proj, gw), res=res)
    d = qt.kernels.fused_gemv(Wo, qt.batch.gnorm_rows(y, proj, gw), res=res)
    assert torch.equal(c, d)
    _close("gnorm + add", to_np(c), O.fused_gemv(to_np(Wo), to_np(y), gnorm=(to_np(proj), to_np(gw)), res=to_np(res)), 2)


def test_no_rows_is_not_an_error(qt, dev):
    W = torch.zeros((64, 1024), dtype=BF16, device=dev)
    x = torch.zeros((0, 1024), dtype=BF16, device=dev)
    assert tuple(qt.kernels.fused_gemv(W, x).shape) == (0, 64)
    assert tuple(qt.batch.rms_rows(x, torch.ones(1024, dtype=BF16, device=dev)).shape) == (0, 1024)


def test_fused_gemv_rejects_bad_arguments(qt, dev):
    W = torch.zeros((64, 1024), dtype=BF16, device=dev)
    x = torch.zeros((2, 1024), dtype=BF16, device=dev)
    with pytest.raises(ValueError):
        qt.kernels.fused_gemv(W, torch.zeros((2, 512), dtype=BF16, device=dev))
    with pytest.raises(ValueError):
        qt.kernels.fused_gemv(W, x, swiglu=True, res=torch.zeros((2, 64), dtype=BF16, device=dev))
    with pytest.raises(TypeError):
        qt.kernels.fused_gemv((W, W), x)
    with pytest.raises(RuntimeError):
        qt.kernels.fused_gemv(torch.zeros((64, 1000), dtype=BF16, device=dev), torch.zeros((2, 1000), dtype=BF16, device=dev))
    with pytest.raises(TypeError):
        qt.kernels.fused_gemv(W.cpu(), x)
    with pytest.raises(IndexError):
        qt.kernels.fused_gemv(torch.zeros((64, 2048), dtype=BF16, device=dev), torch.zeros((2, 2048), dtype=BF16, device=dev),
                              gnorm=(torch.zeros((2, PW), dtype=BF16, device=dev),))
    with pytest.raises(ValueError):                               # rows that are not contiguous are refused in any number of dimensions
        qt.kernels.fused_gemv(W, torch.zeros((1, 2, 2048), dtype=BF16, device=dev)[..., :1024])


def test_row_blocks_are_taken_in_any_shape(qt, dev):
    """a residual and the rows of gated_norm count by their elements: [2 M, N / 2] is [M, N], [S * 16, 128] is [S, 2048]"""
    g = torch.Generator().manual_seed(13)
    W, x = to_dev(rand_bf(g, (64, 1024), 0.03), dev, BF16), to_dev(rand_bf(g, (3, 1024), 1.0), dev, BF16)
    res = to_dev(rand_bf(g, (3, 64), 1.0), dev, BF16)
    assert torch.equal(qt.kernels.fused_gemv(W, x, res=res.reshape(6, 32)), qt.kernels.fused_gemv(W, x, res=res))
    y, proj = to_dev(rand_bf(g, (3, 2048), 1.0), dev, BF16), to_dev(rand_bf(g, (3, PW), 1.0), dev, BF16)
    gw = torch.ones(128, device=dev)
    want = qt.prefill.gated_norm(y, proj, gw)
    assert torch.equal(qt.prefill.gated_norm(y.reshape(48, 128), proj, gw), want)
    assert torch.equal(qt.prefill.gated_norm(y.reshape(3, 16, 128), proj, gw), want)


def test_eps_is_what_float_takes_and_only_where_it_is_used(qt, dev):
    W, x = torch.ones((64, 1024), dtype=BF16, device=dev), torch.ones((2, 1024), dtype=BF16, device=dev)
    want = qt.kernels.fused_gemv(W, x, nw=x[0], eps=0.5)
    check_tensors_equal("eps as text", qt.kernels.fused_gemv(W, x, nw=x[0], eps="0.5"), want)
    check_tensors_equal("no prologue", qt.kernels.fused_gemv(W, x, eps=None), qt.kernels.fused_gemv(W, x))
    with pytest.raises(TypeError):
        qt.kernels.fused_gemv(W, x, nw=x[0], eps=None)


# the model's projections; row counts at the edges of every row block and of the rules that choose a kernel or a tile
@pytest.mark.parametrize("N,K,kind", [(8224, 1024, "rms"), (7168, 1024, "swiglu"), (5120, 1024, "rms"), (1024, 2048, "add"), (1024, 3584, "add")])
def test_a_row_has_the_same_bits_wherever_it_stands(qt, dev, N, K, kind):
    """real-valued rows, so that another order of summation shows: a row's product depends neither on its place in the batch nor (up
    to 64 rows, the wide projections at any number) on how many rows there are"""
    g = torch.Generator().manual_seed(N + K)
    M = 264 if K == 1024 else 64
    W = (torch.randn((N, K), generator=g) * K ** -0.5).to(BF16).to(dev)
    x, nw = torch.randn((M, K), generator=g).to(BF16).to(dev), (1 + 0.1 * torch.randn(K, generator=g)).to(BF16).to(dev)
    res = torch.randn((M, N), generator=g).to(BF16).to(dev)
    f = lambda i: qt.kernels.fused_gemv(W, x[i], nw=nw if kind != "add" else None, res=res[i] if kind == "add" else None, swiglu=kind == "swiglu")
    want = f(torch.arange(M, device=dev))
    for m in (1, 3, 5, 16, 17, 32, 33, 48, 49, 64, 65, 80, 96, 97, 128, 129, 200):
        if m <= M:
            i = torch.randperm(M, generator=g)[:m].to(dev)
            check_tensors_equal(f"{m} rows", f(i), want[i])
