"""Softmax-CE with the rows over many workgroups, at the edges of its lane
groups, label forms and row counts, against float64."""
import ctypes

import numpy as np
import pytest

from tinytorch_amd.hip import DevBuf, check

pytestmark = pytest.mark.gpu


def _ref(x, y):
    x64 = x.astype(np.float64)
    p = np.exp(x64 - x64.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    ok = (y >= 0) & (y < x.shape[1])
    py = np.where(ok, p[np.arange(len(y)), np.where(ok, y, 0)], 0.0)
    seed = p.copy()
    seed[np.arange(len(y))[ok], y[ok]] -= 1.0
    return p, seed / len(y), -np.log(np.maximum(py, 1e-12))


@pytest.mark.parametrize("rows,cols", [(1, 1), (257, 10), (256, 17), (600, 32), (513, 33), (3072, 64),
                                       (3073, 65), (5, 128), (40, 129), (300, 255), (33, 256),
                                       (65, 257), (9, 1000), (20000, 10), (3073, 1), (600, 2),
                                       (4097, 4), (300, 5), (3075, 8), (257, 9)])
def test_softmax_ce_rows(tlib, rows, cols):
    """Every group width (1, 2, 16, 32, 64 lanes, a wavefront) and label form (two
    byte arrays in the arguments, device memory); fp32 exponentials and sums
    of `cols` terms stay within 1e-5 of float64."""
    from tinytorch_amd.torch_py import Node
    rng = np.random.default_rng(rows * 1000 + cols)
    x = (rng.standard_normal((rows, cols)) * 3).astype(np.float32)
    y = rng.integers(0, cols, rows).astype(np.int32)
    if rows > 4:
        y[1], y[3] = -1, cols  # labels outside: no column, the clamped loss
    p64, s64, l64 = _ref(x, y)
    X = Node.leaf(x)
    loss = X.softmax_ce(y)
    loss.backward(None)
    np.testing.assert_allclose(loss.probs(), p64, rtol=1e-5, atol=1e-7)
    # p_y - 1 cancels: the probability's own error, about 4 ulp of 1 (expf,
    # the sum, the division), stays as 2.4e-7 of the seed's scale
    np.testing.assert_allclose(X.grad(), s64, rtol=1e-5, atol=4e-7 / rows)
    np.testing.assert_allclose(loss.value(), [l64.mean()], rtol=1e-5)
    loss.backward(None)  # the kept seed, added
    np.testing.assert_allclose(X.grad(), 2 * s64, rtol=1e-5, atol=8e-7 / rows)
    # the device entry, its mean added in the order of the row losses
    dx, dl = DevBuf.from_np(x), DevBuf.from_np(y)
    pr, se, me, lo = DevBuf(x.size), DevBuf(x.size), DevBuf(1), DevBuf(rows)
    sc = ctypes.c_float(1.0 / rows)
    check(tlib.tt_k_softmax_ce(dx.ptr, dl.ptr, pr.ptr, lo.ptr, se.ptr, rows, cols, sc), "ce")
    np.testing.assert_allclose(lo.to_np((rows,)), l64, rtol=1e-5, atol=1e-5)
    if rows <= 8192:
        check(tlib.tt_k_softmax_ce_mean(dx.ptr, dl.ptr, pr.ptr, me.ptr, se.ptr, rows, cols, sc), "mean")
        check(tlib.tt_k_ce_mean_rows(lo.ptr, lo.ptr, rows), "mean of the rows")
        assert me.to_np((1,))[0] == lo.to_np((rows,))[0]
    for n in (loss, X):
        n.release()


def test_softmax_small_rows(tlib):
    """Rows of up to 64 columns by groups of lanes, with a row of -inf."""
    rng = np.random.default_rng(3)
    for rows, cols in ((1, 10), (17, 16), (5, 17), (100, 64), (3, 1), (513, 2), (257, 4), (9, 5),
                       (260, 8), (18, 9)):
        x = rng.standard_normal((rows, cols)).astype(np.float32)
        x[rows // 2] = -np.inf
        d, y = DevBuf.from_np(x), DevBuf(x.size)
        check(tlib.tt_k_softmax_fwd(d.ptr, y.ptr, rows, cols), "softmax")
        got = y.to_np(x.shape)
        assert np.all(got[rows // 2] == np.float32(1.0) / np.float32(cols))
        keep = np.arange(rows) != rows // 2
        e = np.exp(x[keep].astype(np.float64) - x[keep].max(1, keepdims=True, initial=-1e30))
        np.testing.assert_allclose(got[keep], e / e.sum(1, keepdims=True), rtol=1e-5)


@pytest.mark.parametrize("rows,cols", [(300, 10), (300, 17), (300, 100), (300, 200), (300, 300),
                                       (3073, 1)])
def test_label_outside_the_columns(tlib, rows, cols):
    """A label past the columns has no probability, whatever the row (of -inf:
    1 / cols in each column), and its loss is log(1e-12) with the same bits
    from every entry; a few of them alone make up the mean here."""
    x = np.zeros((rows, cols), np.float32)
    x[:2] = -np.inf
    x[2:, 0] = 200.0  # loss 0 beside those rows
    y = np.zeros(rows, np.int32)
    y[:3] = (cols, cols + 1, -1)
    dx, dl = DevBuf.from_np(x), DevBuf.from_np(y)
    pr, se, me, lo = DevBuf(x.size), DevBuf(x.size), DevBuf(1), DevBuf(rows)
    sc = ctypes.c_float(1.0)
    check(tlib.tt_k_softmax_ce(dx.ptr, dl.ptr, pr.ptr, lo.ptr, se.ptr, rows, cols, sc), "ce")
    got = lo.to_np()
    np.testing.assert_allclose(got[:3], -np.log(1e-12), rtol=1e-6)
    assert np.all(got[3:] == 0.0)
    np.testing.assert_array_equal(pr.to_np((rows, cols))[:2], np.float32(1.0) / np.float32(cols))
    np.testing.assert_array_equal(se.to_np((rows, cols))[:3], pr.to_np((rows, cols))[:3])
    check(tlib.tt_k_softmax_ce_mean(dx.ptr, dl.ptr, pr.ptr, me.ptr, se.ptr, rows, cols, sc), "mean")
    check(tlib.tt_k_ce_mean_rows(lo.ptr, lo.ptr, rows), "mean of the rows")
    assert me.to_np()[0] == lo.to_np()[0]


def test_rows_past_one_launch(tlib):
    """2^28 rows and more by 16 lanes a row are 2^32 work items, which one
    launch does not take: 19 GB of logits and probabilities, all rows alike but
    one on each side of every piece's edge (2^26 rows) and the last."""
    rows, cols = 2 ** 28 + 3, 9
    odd = sorted({k * 2 ** 26 + d for k in range(1, 5) for d in (-1, 0)} | {0, rows - 1})
    x, y = DevBuf(rows * cols), DevBuf(rows * cols)
    x.fill(1.0)
    y.fill(7.0)
    row = np.arange(cols, dtype=np.float32)
    for r in odd:
        check(tlib.tth_h2d(x.ptr + 4 * r * cols, row.ctypes.data, row.nbytes), "h2d")
    e = np.exp(row.astype(np.float64))
    p_odd, p_rest = e / e.sum(), np.full(cols, 1 / cols)

    def rows_of(buf, r, n=cols):
        out = np.empty(n, np.float32)
        check(tlib.tth_d2h(out.ctypes.data, buf.ptr + 4 * r * n, out.nbytes), "d2h")
        return out

    def probabilities(buf):
        for r in odd + [1, 2 ** 26 + 1, rows - 2]:
            np.testing.assert_allclose(rows_of(buf, r), p_odd if r in odd else p_rest, rtol=1e-5)

    check(tlib.tt_k_softmax_fwd(x.ptr, y.ptr, rows, cols), "softmax")
    probabilities(y)
    lab, lo, se = DevBuf(rows, np.int32), DevBuf(rows), DevBuf(rows * cols)
    lab.fill(0.0)  # class 0
    y.fill(7.0)
    check(tlib.tt_k_softmax_ce(x.ptr, lab.ptr, y.ptr, lo.ptr, se.ptr, rows, cols,
                               ctypes.c_float(0.5)), "ce")
    probabilities(y)
    for r in odd + [rows - 2]:
        p = p_odd if r in odd else p_rest
        np.testing.assert_allclose(rows_of(lo, r, 1), [-np.log(p[0])], rtol=1e-5)
        np.testing.assert_allclose(rows_of(se, r), 0.5 * (p - np.eye(cols)[0]), rtol=1e-5, atol=4e-7)


@pytest.mark.parametrize("rows,cols", [(40, 10), (513, 10), (700, 70)])
@pytest.mark.parametrize("what", ["logits", "gradient", "stepped"])
def test_second_backward_has_the_forward_seed(tlib, rows, cols, what):
    """Between two backward passes the host writes the logits or their
    gradient, or a step changes them in place: the second pass still gives the
    forward's seed (fp32: the bounds of test_softmax_ce_rows)."""
    from tinytorch_amd.torch_py import LIB, Node
    rng = np.random.default_rng(rows + cols)
    x = (rng.standard_normal((rows, cols)) * 3).astype(np.float32)
    y = rng.integers(0, cols, rows).astype(np.int32)
    s64 = _ref(x, y)[1]
    X = Node.leaf(x)
    loss = X.softmax_ce(y)
    loss.backward(None)
    n = rows * cols
    if what == "logits":
        np.ctypeslib.as_array(LIB.tt_data(LIB.ag_value(X.ptr)), shape=(n,))[:] = 1
    elif what == "stepped":
        X.sgd_step(1e3)
    else:
        np.ctypeslib.as_array(LIB.tt_data(LIB.ag_grad(X.ptr)), shape=(n,))[:] = 5
    loss.backward(None)
    first = 5.0 if what == "gradient" else s64
    np.testing.assert_allclose(X.grad(), first + s64, rtol=1e-5,
                               atol=4e-7 if what == "gradient" else 8e-7 / rows)
    loss.backward(None)
    np.testing.assert_allclose(X.grad(), first + 2 * s64, rtol=1e-5,
                               atol=8e-7 if what == "gradient" else 1.2e-6 / rows)
    for node in (loss, X):
        node.release()
