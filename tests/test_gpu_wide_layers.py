"""Wide matmul layers: bias and relu in the GEMM's stores, the padded
activations a recipe, the weight gradient from the unpadded input."""
import ctypes

import numpy as np
import pytest

from tinytorch_amd.hip import DevBuf, check

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(31)


@pytest.mark.parametrize("M,N,K", [(1000, 1024, 300),   # two 64x64 tiles a CU
                                   (512, 1024, 512),    # one a CU
                                   (513, 2051, 300),    # rows of C off 16 bytes
                                   (2048, 2048, 130),   # 128x128 tiles
                                   (300, 1100, 900),    # split K: the reduction's epilogue
                                   (2049, 1024, 150)])  # two GEMMs: a pass of its own
def test_gemm_bias_relu(tlib, M, N, K):
    """Bit for bit the product (tt_k_gemm), then bias, then relu."""
    A = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    b = rng.uniform(-1, 1, N).astype(np.float32)
    dA, dB, db = DevBuf.from_np(A), DevBuf.from_np(B), DevBuf.from_np(b)
    C, R, P = DevBuf(M * N), DevBuf(M * N), DevBuf(M * N)
    vp = ctypes.c_void_p
    tlib.ttk_gemm_bias_relu.argtypes = [ctypes.c_int] * 3 + [vp] * 5
    rc = tlib.ttk_gemm_bias_relu(M, N, K, dA.ptr, dB.ptr, db.ptr, C.ptr, R.ptr)
    if 2 * M * N * K < 2 ** 29:
        assert rc == 1
        return
    check(rc, "bias_relu")
    check(tlib.tt_k_gemm(M, N, K, dA.ptr, K, 0, dB.ptr, N, 0, P.ptr, N), "gemm")
    want = P.to_np((M, N)) + b
    assert np.array_equal(C.to_np((M, N)), want)
    assert np.array_equal(R.to_np((M, N)), np.where(want > 0, want, np.float32(0)))


@pytest.mark.parametrize("M,N", [(1, 1), (63, 17), (64, 16), (257, 33), (1000, 10)])
def test_colsum(tlib, M, N):
    g = rng.standard_normal((M, N)).astype(np.float32)
    d, o = DevBuf.from_np(g), DevBuf(N)
    tlib.ttk_colsum.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_int] * 2
    check(tlib.ttk_colsum(d.ptr, o.ptr, M, N), "colsum")
    # fp32 sums of M terms in a tree of depth log2(64) over M / 64 terms
    np.testing.assert_allclose(o.to_np((N,)), g.astype(np.float64).sum(0), rtol=0,
                               atol=2e-7 * np.sqrt(M) * np.abs(g).max() * 4)


@pytest.mark.parametrize("peek", ["none", "padded", "write"])
def test_wide_mlp_step(tlib, peek):
    """A step of a wide MLP against float64: the padded activations unread,
    read in between, or changed by the host through the pinned mirror (the
    weight gradient is then of the changed ones)."""
    from tinytorch_amd.torch_py import Node, Tensor
    B, D, H, O = 700, 400, 1030, 512
    x = rng.uniform(0, 1, (B, D)).astype(np.float32)
    w1 = (rng.standard_normal((D + 1, H)) * 0.05).astype(np.float32)
    w2 = (rng.standard_normal((H + 1, O)) * 0.05).astype(np.float32)
    g = rng.standard_normal((B, O)).astype(np.float32)
    X, W1, W2 = Node.leaf(x, False), Node.leaf(w1), Node.leaf(w2)
    p1 = X.padones()
    h = p1.matmul(W1).relu()
    p2 = h.padones()
    y = p2.matmul(W2)
    y64h = x.astype(np.float64) @ w1[:-1] + w1[-1]
    h64 = np.maximum(y64h, 0)
    a64 = np.c_[h64, np.ones(B)]
    if peek != "none":
        got = p2.value()
        np.testing.assert_allclose(got, a64, rtol=1e-4, atol=1e-4)
    if peek == "write":
        from tinytorch_amd.torch_py import LIB
        t = LIB.ag_value(p2.ptr)
        n = B * (H + 1)
        buf = np.ctypeslib.as_array(LIB.tt_data(t), shape=(n,))
        buf[:] = buf * 2
        a64 = a64 * 2
    y.backward(g)
    np.testing.assert_allclose(W2.grad(), a64.T @ g, rtol=1e-4, atol=2e-3)
    # the relu's side at the GPU's own values: one of 700 x 1030 within rounding
    # of 0 moves a whole term of the sums
    d = (g.astype(np.float64) @ w2.T)[:, :-1] * (h.value() > 0)
    np.testing.assert_allclose(W1.grad(), np.c_[x, np.ones(B)].T.astype(np.float64) @ d, rtol=1e-3,
                               atol=5e-3)
    np.testing.assert_allclose(p2.grad(), g.astype(np.float64) @ w2.T, rtol=1e-4, atol=1e-3)
    for node in (y, p2, h, p1, X, W1, W2):
        node.release()
