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
                                   (2049, 1024, 150),   # a last round of a few tiles
                                   (2049, 1024, 1000)])  # two GEMMs: a pass of its own
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


def _host(node):
    """The host's pointer to a node's value, as a program writes through it."""
    from tinytorch_amd.torch_py import LIB
    t = LIB.ag_value(node.ptr)
    return np.ctypeslib.as_array(LIB.tt_data(t), shape=(int(LIB.tt_numel(t)),))


# M x K of the padded value and N: one that is left unwritten with a GEMM past
# and below the paired kernel's sizes, a narrow one, a classifier
@pytest.mark.parametrize("B,D,H,O", [(700, 400, 1030, 512), (700, 400, 1030, 64),
                                     (40, 30, 50, 60), (40, 30, 50, 10)])
@pytest.mark.parametrize("when", ["source", "padded", "padded, read", "input", "source first",
                                  "padded first"])
def test_padded_value_is_the_forward_one(tlib, B, D, H, O, when):
    """A padones node's value is its input as it was when the node was made:
    the host writing that input afterwards changes nothing, the host writing
    the padded value itself changes the products and weight gradients formed
    with it later.  Against float64 (fp32 sums of at most 1031 products of
    order 1 and of 700 of order 0.5: a few 1e-5 absolute)."""
    from tinytorch_amd.torch_py import Node
    x = rng.uniform(0, 1, (B, D)).astype(np.float32)
    w1 = (rng.standard_normal((D + 1, H)) * 0.05).astype(np.float32)
    w2 = (rng.standard_normal((H + 1, O)) * 0.05).astype(np.float32)
    g = rng.standard_normal((B, O)).astype(np.float32)
    X, W1, W2 = Node.leaf(x, False), Node.leaf(w1), Node.leaf(w2)
    one = np.ones((B, 1))
    x64 = np.c_[x.astype(np.float64), one]
    a64 = np.c_[np.maximum(x64 @ w1, 0), one]
    p1 = X.padones()
    h = p1.matmul(W1).relu()
    p2 = h.padones()
    if when == "source first":
        _host(h)[:] *= 2
    if when == "padded first":
        _host(p2)[:] *= 2
        a64 = a64 * 2
    y = p2.matmul(W2)
    keep = []
    if when in ("source first", "padded first"):
        np.testing.assert_allclose(y.value(), a64 @ w2, rtol=1e-4, atol=1e-3)
    if when == "source":
        _host(h)[:] *= 2
    if when == "input":
        _host(X)[:] *= 2
    if when.startswith("padded") and when != "padded first":
        _host(p2)[:] *= 2
        a64 = a64 * 2
    if when == "padded, read":
        keep.append(p2 * 1.0)  # the host's copy goes to the device before the backward
        np.testing.assert_allclose(keep[0].value(), a64, rtol=1e-4, atol=1e-4)
    y.backward(g)
    np.testing.assert_allclose(W2.grad(), a64.T @ g, rtol=1e-4, atol=2e-3)
    if not when.startswith("source"):  # (the relu's backward reads its output)
        d = (g.astype(np.float64) @ w2.T)[:, :-1] * (h.value() > 0)
        np.testing.assert_allclose(W1.grad(), x64.T @ d, rtol=1e-3, atol=5e-3)
    for node in keep + [y, p2, h, p1, X, W1, W2]:
        node.release()


@pytest.mark.parametrize("M,K,N", [(600, 500, 512), (600, 500, 48), (50, 40, 48), (50, 40, 10)])
def test_padded_leaf_stepped_between_backwards(tlib, M, K, N):
    """A leaf stepped in place between two backward passes over one graph: the
    second weight gradient is of the padded value the forward made."""
    from tinytorch_amd.torch_py import Node
    x = rng.uniform(0, 1, (M, K)).astype(np.float32)
    w = (rng.standard_normal((K + 1, N)) * 0.05).astype(np.float32)
    g = rng.standard_normal((M, N)).astype(np.float32)
    X, W = Node.leaf(x), Node.leaf(w)
    p = X.padones()
    y = p.matmul(W)
    y.backward(g)
    X.sgd_step(0.5)
    assert np.abs(X.value() - x).max() > 0.01
    y.backward(g)
    # the second pass adds to the first
    want = 2 * np.c_[x.astype(np.float64), np.ones(M)].T @ g
    np.testing.assert_allclose(W.grad(), want, rtol=1e-4, atol=4e-3)
    for node in (y, p, X, W):
        node.release()


def test_softmax_ce_padded_source_written(tlib):
    """The classifier whose input gradients were formed with the softmax-CE:
    the relu output written by the host before the backward leaves the weight
    gradient that of the padded value."""
    from tinytorch_amd.torch_py import Node
    B, D, H, C = 64, 96, 128, 10
    x = rng.uniform(0, 1, (B, D)).astype(np.float32)
    w1 = (rng.standard_normal((D + 1, H)) * 0.1).astype(np.float32)
    w2 = (rng.standard_normal((H + 1, C)) * 0.1).astype(np.float32)
    lab = rng.integers(0, C, B)
    X, W1, W2 = Node.leaf(x, False), Node.leaf(w1), Node.leaf(w2)
    p1 = X.padones()
    h = p1.matmul(W1).relu()
    p2 = h.padones()
    z = p2.matmul(W2)
    loss = z.softmax_ce(lab)
    a64 = np.c_[np.maximum(np.c_[x.astype(np.float64), np.ones(B)] @ w1, 0), np.ones(B)]
    e = np.exp(a64 @ w2)
    seed = e / e.sum(1, keepdims=True)
    seed[np.arange(B), lab] -= 1
    _host(h)[:] = 3
    loss.backward()
    np.testing.assert_allclose(W2.grad(), a64.T @ (seed / B), rtol=1e-4, atol=1e-5)
    for node in (loss, z, p2, h, p1, X, W1, W2):
        node.release()
