"""The 128x128 direct-load tiles and the plan of large plain GEMMs (a kernel,
a split, or two GEMMs) against float64, at the GEMM bar max|err| / (sqrt(K) *
max|A| * max|B|) <= 1e-4, far above fp32 sums in any order."""
import ctypes

import numpy as np
import pytest

from tinytorch_amd.hip import DevBuf, check

pytestmark = pytest.mark.gpu
rng = np.random.default_rng(77)
TOL = 1e-4


def _run(tlib, M, N, K, ta, tb, fn="tt_k_gemm"):
    A = rng.uniform(-1, 1, (K, M) if ta else (M, K)).astype(np.float32)
    B = rng.uniform(-1, 1, (N, K) if tb else (K, N)).astype(np.float32)
    dA, dB, dC = DevBuf.from_np(A), DevBuf.from_np(B), DevBuf(M * N + 64)
    dC.fill(7.0)  # what lies past C stays as it is
    check(getattr(tlib, fn)(M, N, K, dA.ptr, M if ta else K, ta, dB.ptr, K if tb else N, tb,
                            dC.ptr, N), fn)
    C = dC.to_np((M * N + 64,))
    assert np.all(C[M * N:] == 7.0)
    a = (A.T if ta else A).astype(np.float64)
    b = (B.T if tb else B).astype(np.float64)
    err = np.abs(C[:M * N].reshape(M, N) - a @ b).max() / np.sqrt(K)
    assert err <= TOL, (M, N, K, ta, tb, err)
    return C[:M * N], (dA, dB)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (128, 128, 32), (127, 129, 31), (129, 127, 33),
                                   (130, 260, 97), (257, 3, 200), (4, 300, 128), (256, 384, 160),
                                   (64, 68, 4)])
def test_ring_tiles(tlib, M, N, K, ta, tb):
    """Every transposition, 4- and 16-byte loads, edges of tiles and of K's
    32-k stages (fewer stages than the ring holds included)."""
    L = tlib
    L.ttk_gemm_large.argtypes = [ctypes.c_int]
    prev = L.ttk_gemm_large(2)
    try:
        _run(tlib, M, N, K, ta, tb)
    finally:
        L.ttk_gemm_large(prev)


@pytest.mark.parametrize("M,N,K,ta,tb", [
    (2049, 1024, 300, 1, 0),    # 2048 rows and one of their own
    (1000, 2049, 512, 0, 1),    # the same in columns
    (1153, 2304, 301, 0, 0),    # 128x128 tiles, a ragged last row of them
    (3329, 2300, 64, 0, 0),     # a second GEMM of a few tile rows
    (300, 700, 2600, 0, 1),     # split K
    (1024, 1024, 256, 1, 1),    # whole tiles, both transposed
])
def test_large_plan(tlib, M, N, K, ta, tb):
    """Each outcome of the plan, and the entry without allocation: the same bits."""
    c, (dA, dB) = _run(tlib, M, N, K, ta, tb)
    out = DevBuf(M * N)
    check(tlib.tt_k_gemm_noalloc(M, N, K, dA.ptr, M if ta else K, ta, dB.ptr, K if tb else N, tb,
                                 out.ptr, N), "noalloc")
    assert np.array_equal(out.to_np((M * N,)), c)
