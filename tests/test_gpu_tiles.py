"""Tile sizes that are no multiple of 64, through the factorisations and solves.

Square matrices are held in tiles rounded up to 64: sizes at the edges of 16 and
64, one tile shorter than its block size, many small tiles, square right-hand
sides, and one matrix too large for that rounding (16-column tiles).  Solutions
against numpy in FP64: cond(A) is O(1) for these matrices, so the relative
error is a few n eps, 1e-12 at most; the large one by its residual
|AX - B| / (|A| |X| n eps), a few at most for a backward stable solve.
"""
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


@pytest.mark.parametrize("n,nb,nrhs", [(1, 16, 1), (17, 17, 17), (63, 128, 1), (65, 200, 70), (96, 128, 8),
                                       (130, 65, 9), (300, 48, 3), (333, 40, 65), (500, 17, 500), (700, 200, 64),
                                       (1000, 1024, 5), (1100, 336, 1)])
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
def test_factor_and_solve(ch, n, nb, nrhs, uplo):
    print("[case] tiles", n, nb, nrhs, uplo, flush=True)
    L = ch.lib
    A = oracle.dplgsy(float(n), FULL, n, 3)
    B = oracle.dplrnt(n, nrhs, 4)
    want = np.linalg.solve(A, B)
    seq = ch.Sequence()
    with ch.Desc.from_array(A.copy(order="F"), nb) as dA, ch.Desc.from_array(B.copy(order="F"), nb) as dB, \
            ch.Desc.from_array(B.copy(order="F"), nb) as dX:
        ch.check(L.CHAMELEON_dposv_Tile_Async(uplo, dA.ptr, dB.ptr, seq.ptr, seq.req))
        ch.check(L.CHAMELEON_dpotrs_Tile_Async(uplo, dA.ptr, dX.ptr, seq.ptr, seq.req))
        ch.check(seq.wait())
        assert oracle.rel_frobenius(dB.to_array(n, nrhs), want) <= 1e-12
        assert oracle.rel_frobenius(dX.to_array(n, nrhs), want) <= 1e-12
        F = dA.to_array(n, n)
        C = np.linalg.cholesky(A)
        F, C = (np.tril(F), C) if uplo == LOWER else (np.triu(F), C.T)
        assert oracle.rel_frobenius(F, C) <= 1e-12
    seq.destroy()


def test_not_positive_definite(ch):
    n, nb = 250, 100
    A = oracle.dplgsy(float(n), FULL, n, 3)
    A[170, 170] = -1.0
    seq = ch.Sequence()
    with ch.Desc.from_array(A.copy(order="F"), nb) as dA:
        ch.lib.CHAMELEON_dpotrf_Tile_Async(LOWER, dA.ptr, seq.ptr, seq.req)
        assert seq.wait() == 171
    seq.destroy()


def test_small_tiles_past_the_rounding(ch):
    n, nb, nrhs = 11600, 16, 3
    print("[case] tiles", n, nb, nrhs, flush=True)
    rng = np.random.default_rng(7)
    A = rng.standard_normal((n, n))
    A = np.asfortranarray(A + A.T)
    A[np.diag_indices(n)] += 4.0 * n
    B = np.asfortranarray(rng.standard_normal((n, nrhs)))
    seq = ch.Sequence()
    with ch.Desc.from_array(A.copy(order="F"), nb) as dA, ch.Desc.from_array(B.copy(order="F"), nb) as dB:
        ch.check(ch.lib.CHAMELEON_dposv_Tile_Async(LOWER, dA.ptr, dB.ptr, seq.ptr, seq.req))
        ch.check(seq.wait())
        X = dB.to_array(n, nrhs)
    r = np.abs(A @ X - B).max(axis=0)
    eps = np.finfo(float).eps
    assert (r <= 4.0 * n * eps * 6.0 * n * np.abs(X).max(axis=0)).all()
    seq.destroy()
