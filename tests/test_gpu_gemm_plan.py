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


MID, RING, DIRECT, SPLIT, ROWS, COLS = range(6)  # ttk_gemm_plan_taken's outcomes


def _taken(L):
    L.ttk_gemm_plan_taken.restype = ctypes.c_long
    return np.array([L.ttk_gemm_plan_taken(i) for i in range(6)])


def _planned(tlib, M, N, K, ta, tb):
    """One GEMM and the entry without allocation, the same bits; the plan's
    outcomes of the first."""
    before = _taken(tlib)
    c, (dA, dB) = _run(tlib, M, N, K, ta, tb)
    got = _taken(tlib) - before
    out = DevBuf(M * N)
    check(tlib.tt_k_gemm_noalloc(M, N, K, dA.ptr, M if ta else K, ta, dB.ptr, K if tb else N, tb,
                                 out.ptr, N), "noalloc")
    assert np.array_equal(out.to_np((M * N,)), c)
    return got


@pytest.mark.parametrize("M,N,K,ta,tb,outcome", [
    (2049, 1024, 300, 1, 0, MID),    # a last round of a few tiles, cheaper than a second GEMM
    (1000, 2049, 512, 0, 1, MID),
    (1153, 2304, 301, 0, 0, MID),
    (3329, 2300, 64, 0, 0, None),    # few k: not planned
    (8000, 7936, 64, 0, 0, None),
    (11499, 3969, 31, 0, 1, None),
    (3329, 2300, 68, 0, 0, RING),    # a ragged last row and column of 128x128 tiles
    (300, 700, 2600, 0, 1, MID),     # few tiles: split K on 64x64 ones
    (1024, 1024, 256, 1, 1, MID),    # whole tiles, both transposed
    (1400, 1200, 4096, 0, 1, SPLIT),
    (1400, 1200, 4095, 1, 0, SPLIT),  # 4-byte loads, a ragged last split
    (4096, 4096, 96, 0, 0, DIRECT),
])
def test_large_plan(tlib, M, N, K, ta, tb, outcome):
    """Each kernel that the plan gives a single GEMM to, and shapes it leaves."""
    got = _planned(tlib, M, N, K, ta, tb)
    assert got.sum() == (outcome is not None) and (outcome is None or got[outcome] == 1), got


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K,cut", [(2049, 1024, 1000, ROWS), (1024, 2049, 1000, COLS),
                                       (2051, 1024, 999, ROWS), (1024, 2051, 999, COLS)])
def test_two_gemms(tlib, M, N, K, cut, ta, tb):
    """The rows or columns past the last full round of tiles as a GEMM of their
    own, from every layout of both operands, 16- and 4-byte loads."""
    got = _planned(tlib, M, N, K, ta, tb)
    assert got[cut] == 1 and got[ROWS] + got[COLS] == 1, got
