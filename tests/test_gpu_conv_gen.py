"""The convolution over channel chunks (conv_gen.hip) against the oracle's
conv2d forward / backward (reference src/ops_spatial.c:71-127,
src/autograd.c:456-553), at the GEMM bar max|err| / (sqrt(K) * max|A| *
max|B|) <= 1e-4, K the summed length: fp32 sums of K products in any order
stay a few ulp * sqrt(K) from the exact one, far below it."""
import ctypes

import numpy as np
import pytest

import orc
from tinytorch_amd.hip import DevBuf, check

rng = np.random.default_rng(909)
TOL = 1e-4

# (N, C, H, W, F, HH, WW, sh, sw, ph, pw)
CASES = [
    (1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0),        # one product
    (3, 8, 7, 7, 32, 3, 3, 1, 1, 1, 1),       # tiles over several images, one whole chunk
    (2, 9, 12, 11, 33, 3, 3, 1, 1, 1, 1),     # a chunk of one channel, a filter block of one
    (2, 17, 5, 61, 40, 3, 5, 1, 1, 1, 2),     # rows of 65 columns: two pieces a row
    (1, 10, 6, 130, 8, 3, 3, 1, 1, 1, 1),     # three pieces a row
    (5, 12, 9, 10, 65, 5, 5, 2, 2, 2, 2),     # stride 2: four residues of 9, 6, 6, 4 taps
    (4, 16, 10, 9, 20, 1, 1, 2, 2, 0, 0),     # residues with no tap: zeros in dX
    (2, 6, 13, 14, 7, 3, 2, 3, 1, 0, 1),      # strides 3 and 1, a 3x2 kernel
    (2, 5, 8, 8, 6, 3, 3, 1, 1, 4, 3),        # padding past the kernel
    (2, 24, 16, 16, 130, 3, 3, 1, 1, 1, 1),   # 130 filters; 128 x 64 weight-gradient tiles
    (20, 33, 19, 17, 31, 3, 3, 1, 1, 0, 1),   # odd image sizes: 4-byte loads of g
    (6, 70, 4, 4, 16, 1, 1, 1, 1, 0, 0),      # 1x1, 70 channels
]


def err(got, ref, K, amax, bmax):
    return np.abs(got.astype(np.float64) - ref).max() / (np.sqrt(K) * amax * bmax)


def _q(case):
    N, C, H, W, F, HH, WW, sh, sw, ph, pw = case
    Ho, Wo = orc.conv_out(H, W, HH, WW, sh, sw, ph, pw)
    return (ctypes.c_int * 13)(*case, Ho, Wo), Ho, Wo


def _lib():
    import tinytorch_amd
    L = tinytorch_amd.lib()
    vp = ctypes.c_void_p
    L.ttk_conv_gen_fwd.argtypes = [vp] * 5 + [vp]
    L.ttk_conv_gen_dx.argtypes = [vp] * 3 + [vp]
    L.ttk_conv_gen_dw.argtypes = [vp] * 4 + [vp]
    L.ttk_conv_gen_force.argtypes = [ctypes.c_int] * 4
    L.ttk_conv_gen_force.restype = None
    L.ttk_conv_route.argtypes = [vp, ctypes.c_int]
    return L


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [-1, 0, 1, 2, 3])
@pytest.mark.parametrize("case", CASES)
def test_conv_gen_vs_oracle(tlib, case, tile):
    N, C, H, W, F, HH, WW, sh, sw, ph, pw = case
    q, Ho, Wo = _q(case)
    L = _lib()
    print("conv gen", case, tile, flush=True)
    x = rng.uniform(-1, 1, (N, C, H, W)).astype(np.float32)
    w = rng.uniform(-1, 1, (F, C, HH, WW)).astype(np.float32)
    b = rng.uniform(-1, 1, F).astype(np.float32)
    g = rng.uniform(-1, 1, (N, F, Ho, Wo)).astype(np.float32)
    dx_, dw_, db_, dg_ = (DevBuf.from_np(a) for a in (x, w, b, g))
    y, r, dX, dW, dB = (DevBuf(n) for n in (g.size, g.size, x.size, w.size, F))
    rdx, rdw, rdb = orc.conv2d_bwd(x, w, g, sh, sw, ph, pw)
    # every tile, and for the weight gradient every tile and split count
    L.ttk_conv_gen_force(tile, 0, -1 if tile < 0 else min(tile, 2), 0 if tile < 1 else tile)
    try:
        if L.ttk_conv_gen_fwd(None, None, None, None, None, q) == 0:
            check(L.ttk_conv_gen_fwd(dx_.ptr, dw_.ptr, db_.ptr, y.ptr, r.ptr, q), "fwd")
            ref = orc.conv2d_fwd(x, w, b, sh, sw, ph, pw)
            got = y.to_np(ref.shape)
            assert err(got, ref, C * HH * WW, 1.0, 1.0) <= TOL
            assert np.array_equal(r.to_np(ref.shape), np.where(got > 0, got, np.float32(0)))
        else:
            assert tile >= 0  # the planner finds a tile for every case here
        if L.ttk_conv_gen_dx(None, None, None, q) == 0:
            check(L.ttk_conv_gen_dx(dg_.ptr, dw_.ptr, dX.ptr, q), "dx")
            assert err(dX.to_np(x.shape), rdx, F * HH * WW, 1.0, 1.0) <= TOL
        else:
            assert tile >= 0
        if L.ttk_conv_gen_dw(None, None, None, None, q) == 0:
            check(L.ttk_conv_gen_dw(dg_.ptr, dx_.ptr, dW.ptr, dB.ptr, q), "dw")
            assert err(dW.to_np(w.shape), rdw, N * Ho * Wo, 1.0, 1.0) <= TOL
            assert err(dB.to_np((F,)), rdb, N * Ho * Wo, 1.0, 1.0) <= TOL
            one = dW.to_np(w.shape)
            check(L.ttk_conv_gen_dw(dg_.ptr, dx_.ptr, dW.ptr, None, q), "dw without db")
            assert np.array_equal(dW.to_np(w.shape), one)  # deterministic
        else:
            assert tile >= 0
    finally:
        L.ttk_conv_gen_force(-1, 0, -1, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[2], CASES[5], CASES[10]])
def test_conv_gen_nonfinite_stays_local(tlib, case):
    """An infinity reaches only the outputs its taps reach: padding, missing
    channels and pixels past the range are products of zeros."""
    N, C, H, W, F, HH, WW, sh, sw, ph, pw = case
    q, Ho, Wo = _q(case)
    L = _lib()
    x = rng.uniform(0.5, 1, (N, C, H, W)).astype(np.float32)
    w = rng.uniform(0.5, 1, (F, C, HH, WW)).astype(np.float32)
    g = rng.uniform(0.5, 1, (N, F, Ho, Wo)).astype(np.float32)
    y, dX, dW = DevBuf(g.size), DevBuf(x.size), DevBuf(w.size)
    bad = x.copy()
    bad[N - 1, C - 1, H - 1, W - 1] = np.inf
    wbad = w.copy()
    wbad[F - 1, C - 1, 0, 0] = np.inf
    gbad = g.copy()
    gbad[N - 1, F - 1, Ho - 1, Wo - 1] = np.inf
    dg_, dx_, dw_ = (DevBuf.from_np(a) for a in (gbad, bad, wbad))
    check(L.ttk_conv_gen_fwd(dx_.ptr, DevBuf.from_np(w).ptr, None, y.ptr, None, q), "fwd")
    tlib.tth_sync()
    assert np.array_equal(np.isfinite(y.to_np(g.shape)),
                          np.isfinite(orc.conv2d_fwd(bad, w, np.zeros(F, np.float32), sh, sw, ph, pw)))
    wd = DevBuf.from_np(w)
    check(L.ttk_conv_gen_dx(dg_.ptr, wd.ptr, dX.ptr, q), "dx")
    xd = DevBuf.from_np(x)
    check(L.ttk_conv_gen_dw(dg_.ptr, xd.ptr, dW.ptr, None, q), "dw")
    rdx, rdw, _ = orc.conv2d_bwd(x, w, gbad, sh, sw, ph, pw)
    assert np.array_equal(np.isfinite(dX.to_np(x.shape)), np.isfinite(rdx))
    assert np.array_equal(np.isfinite(dW.to_np(w.shape)), np.isfinite(rdw))
    xd2, wd2 = DevBuf.from_np(x), DevBuf.from_np(wbad)
    check(L.ttk_conv_gen_fwd(xd2.ptr, wd2.ptr, None, y.ptr, None, q), "fwd")
    assert np.array_equal(np.isfinite(y.to_np(g.shape)), np.isfinite(
        orc.conv2d_fwd(x, wbad, np.zeros(F, np.float32), sh, sw, ph, pw)))


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("case", [CASES[k] for k in (1, 2, 3, 5, 6, 7, 8, 9)])
def test_conv_gen_dx_nonfinite_weight(tlib, case, bad):
    """The input gradient adds only the taps that reach an element: an infinite
    or NaN weight changes the elements that it reaches, and none beside the
    border that it does not (the padding is no product of its)."""
    N, C, H, W, F, HH, WW, sh, sw, ph, pw = case
    q, Ho, Wo = _q(case)
    L = _lib()
    w = rng.uniform(0.5, 1, (F, C, HH, WW)).astype(np.float32)
    w[F - 1, C - 1, 0, 0] = bad
    g = rng.uniform(0.5, 1, (N, F, Ho, Wo)).astype(np.float32)
    x = np.zeros((N, C, H, W), np.float32)
    dX, gd, wd = DevBuf(x.size), DevBuf.from_np(g), DevBuf.from_np(w)
    check(L.ttk_conv_gen_dx(gd.ptr, wd.ptr, dX.ptr, q), "dx")
    ref, got = orc.conv2d_bwd(x, w, g, sh, sw, ph, pw)[0], dX.to_np(x.shape)
    fin = np.isfinite(ref)
    assert not fin.all() and fin.any()
    assert np.array_equal(np.isfinite(got), fin)
    assert err(got[fin], ref[fin], F * HH * WW, 1.0, 1.0) <= TOL


def test_conv_route():
    """Which kernel a convolution takes (no GPU needed)."""
    L = _lib()

    def route(case, what):
        return L.ttk_conv_route(_q(case)[0], what)
    slab, chunk = 1, 2
    config = (128, 32, 16, 16, 64, 3, 3, 1, 1, 1, 1)
    assert [route(config, k) for k in range(3)] == [slab] * 3
    assert route((128, 3, 32, 32, 32, 3, 3, 1, 1, 1, 1), 0) == slab
    big = (32, 64, 56, 56, 128, 3, 3, 1, 1, 1, 1)
    assert [route(big, k) for k in range(3)] == [chunk] * 3
    assert [route((50, 24, 45, 37, 40, 5, 5, 2, 2, 2, 2), k) for k in range(3)] == [chunk] * 3
    assert route((64, 8, 30, 30, 200, 3, 3, 1, 1, 1, 1), 2) == 0  # few channels: GEMM + col2im
    prev = L.tth_conv_lds(0)
    try:
        assert [route(config, k) for k in range(3)] == [0] * 3
        assert [route(big, k) for k in range(3)] == [0] * 3
    finally:
        L.tth_conv_lds(prev)


@pytest.mark.parametrize("case,routes,direct", [
    # the direct kernels of the forward and the weight gradient, the input
    # gradient's (0: GEMM + col2im); whether a forward, a forward and weight
    # gradient run direct
    ((50, 24, 45, 37, 40, 5, 5, 2, 2, 2, 2), (2, 2, 2), (1, 1)),
    ((37, 9, 55, 55, 13, 1, 1, 1, 1, 0, 0), (1, 1, 1), (1, 1)),    # 1x1: slab 10.6 us, chunks 11.7
    ((14, 14, 18, 62, 6, 1, 1, 1, 1, 0, 0), (1, 1, 1), (1, 1)),    # 5.7 / 7.6
    ((5, 119, 9, 15, 36, 5, 5, 2, 2, 1, 2), (2, 2, 0), (0, 0)),    # few tiles, 15 chunks: GEMM 17.7, chunks 43.5
    ((1, 59, 23, 33, 9, 5, 5, 2, 2, 2, 2), (2, 2, 2), (0, 0)),     # 11.6 / 29.2
    ((3, 109, 25, 47, 4, 5, 5, 2, 2, 2, 2), (2, 2, 2), (0, 0)),    # 22.1 / 45.2
    ((12, 89, 11, 43, 39, 1, 1, 2, 2, 0, 0), (2, 1, 0), (0, 0)),   # 11.1 / 15.1
])
def test_conv_direct(case, routes, direct):
    """Where the chunks would be the slower choice the GEMM or slab kernels
    stay (no GPU needed)."""
    L = _lib()
    L.ttk_conv_direct.argtypes = [ctypes.c_void_p, ctypes.c_int]
    q = _q(case)[0]
    assert tuple(L.ttk_conv_route(q, k) for k in range(3)) == routes
    assert tuple(L.ttk_conv_direct(q, k) for k in range(2)) == direct


@pytest.mark.gpu
@pytest.mark.parametrize("case", [(5, 119, 9, 15, 36, 5, 5, 2, 2, 1, 2),   # GEMM throughout
                                  (1, 59, 23, 33, 9, 5, 5, 2, 2, 2, 2),    # GEMM, dX by chunks
                                  (12, 89, 11, 43, 39, 1, 1, 2, 2, 0, 0),
                                  (14, 14, 18, 62, 6, 1, 1, 1, 1, 0, 0)])  # slab
@pytest.mark.parametrize("train", [0, 1])
def test_conv_mixed_routes(tlib, case, train):
    """A layer whose products take different paths, with and without its weight
    gradient (a forward that keeps its im2col matrix or not)."""
    from tinytorch_amd.torch_py import Node
    N, C, H, W, F, HH, WW, sh, sw, ph, pw = case
    _, Ho, Wo = _q(case)
    x = rng.uniform(-1, 1, (N, C, H, W)).astype(np.float32)
    w = rng.uniform(-1, 1, (F, C, HH, WW)).astype(np.float32)
    b = rng.uniform(-1, 1, F).astype(np.float32)
    g = rng.uniform(-1, 1, (N, F, Ho, Wo)).astype(np.float32)
    X, Wn, Bn = Node.leaf(x), Node.leaf(w, bool(train)), Node.leaf(b, bool(train))
    y = X.conv2d(Wn, Bn, (sh, sw), (ph, pw))
    y.backward(g)
    rdx, rdw, rdb = orc.conv2d_bwd(x, w, g, sh, sw, ph, pw)
    K = C * HH * WW
    assert err(y.value(), orc.conv2d_fwd(x, w, b, sh, sw, ph, pw), K, 1.0, 1.0) <= TOL
    assert err(X.grad(), rdx, F * HH * WW, 1.0, 1.0) <= TOL
    if train:
        assert err(Wn.grad(), rdw, N * Ho * Wo, 1.0, 1.0) <= TOL
        assert err(Bn.grad(), rdb, N * Ho * Wo, 1.0, 1.0) <= TOL
    for node in (y, X, Wn, Bn):
        node.release()
