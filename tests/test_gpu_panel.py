"""The fused panel kernel at the edges of its work split.

Column blocks per tile (the tile size over 64): 1 (the chain alone), 2 (no
block between the chain's), 3 and 4 (the first units of a higher level), 17
(more units of the diagonal tile than the seven of the smallest split, and with
seven tiles below fewer workgroups than units); a last tile that ends inside,
at the edge of and one past a 16-column step.  Factor against the oracle to the
relative 1e-12 of the other FP64 factor tests (the error of a backward-stable
Cholesky of these matrices is a few n eps / 100), non-positive pivots at the
first and last column of a 16-column step, a 64-column block and a tile.
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

LOWER, UPPER, FULL = 122, 121, 123


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.init()
    yield ch


def _p(a):
    return ctypes.c_void_p(a.ctypes.data)


@pytest.mark.parametrize("n,nb", [(64, 64), (129, 64), (128, 128), (500, 128), (577, 192), (1040, 256), (1041, 256),
                                  (2048, 512), (2575, 512), (2300, 1088), (8300, 1088)])
def test_factor(ch, n, nb):
    print("[case] panel", n, nb, flush=True)
    ch.set_param(ch.TILE_SIZE, nb)
    A = oracle.dplgsy(float(n), FULL, n, 7)
    upper = np.triu(A, 1).copy()
    ref = A.copy(order="F")
    assert ch.lib.CHAMELEON_dpotrf(LOWER, n, _p(A), n) == 0
    oracle.use_blas(True)
    try:
        assert oracle.dpotrf(LOWER, ref, n, nb) == 0
    finally:
        oracle.use_blas(False)
    assert oracle.rel_frobenius(np.tril(A), np.tril(ref)) <= 1e-12
    assert np.array_equal(np.triu(A, 1), upper)


@pytest.mark.parametrize("j", [0, 15, 16, 63, 64, 127, 255, 256, 319, 511, 512, 639])
def test_first_bad_pivot(ch, j):
    """One diagonal entry made negative: the factorisation stops there."""
    n, nb = 640, 256
    print("[case] pivot", j, flush=True)
    ch.set_param(ch.TILE_SIZE, nb)
    A = oracle.dplgsy(float(n), FULL, n, 51)
    A[j, j] = -1.0
    assert ch.lib.CHAMELEON_dpotrf(LOWER, n, _p(A), n) == j + 1
    A = oracle.dplgsy(float(n), FULL, n, 51)
    assert ch.lib.CHAMELEON_dpotrf(LOWER, n, _p(A), n) == 0
