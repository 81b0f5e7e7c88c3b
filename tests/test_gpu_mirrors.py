"""Matrices of one tiling whose device copies are padded differently.

A square matrix is held in tiles rounded up to 64 when there is memory for it and
to 16 otherwise, so A, B and X of one call may have either.  Every combination,
with square right-hand sides: solutions against numpy (cond(A) is O(1): a few n
eps, 1e-12), and the backward error of integer matrices, whose sums are exact
(only the quotient rounds, 1e-14).
"""
import ctypes
import itertools
import os

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

LOWER, FULL = 122, 123


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.init()
    ch.lib.CHAMAMD_Backward_Error.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                                              ctypes.POINTER(ctypes.c_double)]
    yield ch


def resident(ch, seq, src, dst, wide):
    """dst <- src on the device, its copy there made with the large or the small padding."""
    if not wide:
        os.environ["CHAMAMD_PAD64"] = "0"
    try:
        ch.check(ch.lib.CHAMELEON_dlacpy_Tile_Async(FULL, src.ptr, dst.ptr, seq.ptr, seq.req))
        ch.check(seq.wait())
    finally:
        os.environ.pop("CHAMAMD_PAD64", None)


COMBINATIONS = list(itertools.product((False, True), repeat=3))


@pytest.mark.parametrize("n,nb", [(300, 100), (70, 200)])
@pytest.mark.parametrize("wide", COMBINATIONS)
def test_fp64_fallback(ch, n, nb, wide):
    print("[case] mirrors", n, nb, wide, flush=True)
    A = oracle.dplgsy(float(n), FULL, n, 3)
    B = oracle.dplrnt(n, n, 4)
    it, berr = ctypes.c_int(), ctypes.c_double()
    seq = ch.Sequence()
    D = ch.Desc
    with D.from_array(A.copy(order="F"), nb) as hA, D.from_array(B.copy(order="F"), nb) as hB, \
            D.alloc(n, n, nb) as dA, D.alloc(n, n, nb) as dB, D.alloc(n, n, nb) as dX:
        for src, dst, w in ((hA, dA, wide[0]), (hB, dB, wide[1]), (hB, dX, wide[2])):
            resident(ch, seq, src, dst, w)
        ch.check(ch.lib.CHAMAMD_dposv_mixed_Tile_Async(LOWER, dA.ptr, dB.ptr, dX.ptr, 0, ctypes.byref(it),
                                                       ctypes.byref(berr), seq.ptr, seq.req))
        ch.check(seq.wait())
        X = dX.to_array(n, n)
        assert np.array_equal(dB.to_array(n, n), B)
    seq.destroy()
    assert it.value == -1
    assert oracle.rel_frobenius(X, np.linalg.solve(A, B)) <= 1e-12


@pytest.mark.parametrize("n,nb", [(300, 100), (70, 200)])
@pytest.mark.parametrize("wide", COMBINATIONS)
def test_backward_error(ch, n, nb, wide):
    print("[case] mirrors, backward error", n, nb, wide, flush=True)
    rng = np.random.default_rng(n)
    A = np.asfortranarray(rng.integers(-9, 10, (n, n)).astype(float))
    S = np.tril(A) + np.tril(A, -1).T
    X = np.asfortranarray(rng.integers(-9, 10, (n, n)).astype(float))
    B = np.asfortranarray(rng.integers(-99, 100, (n, n)).astype(float))
    R = np.abs(B - S @ X).max(axis=0)
    want = (R / (np.abs(S).sum(axis=1).max() * np.abs(X).max(axis=0) * n * 2.0 ** -53)).max()
    be = ctypes.c_double()
    seq = ch.Sequence()
    D = ch.Desc
    with D.from_array(A, nb) as hA, D.from_array(X, nb) as hX, D.from_array(B, nb) as hB, \
            D.alloc(n, n, nb) as dA, D.alloc(n, n, nb) as dX, D.alloc(n, n, nb) as dB:
        for src, dst, w in ((hA, dA, wide[0]), (hX, dX, wide[1]), (hB, dB, wide[2])):
            resident(ch, seq, src, dst, w)
        assert ch.lib.CHAMAMD_Backward_Error(LOWER, dA.ptr, dX.ptr, dB.ptr, ctypes.byref(be)) == 0
    seq.destroy()
    assert abs(be.value - want) <= 1e-14 * want, (be.value, want)


@pytest.mark.parametrize("wide", COMBINATIONS)
def test_factor_and_solve(ch, wide):
    n, nb = 333, 40
    print("[case] mirrors, dposv and dpotrs", wide, flush=True)
    A = oracle.dplgsy(float(n), FULL, n, 3)
    B = oracle.dplrnt(n, n, 4)
    want = np.linalg.solve(A, B)
    seq = ch.Sequence()
    D = ch.Desc
    with D.from_array(A.copy(order="F"), nb) as hA, D.from_array(B.copy(order="F"), nb) as hB, \
            D.alloc(n, n, nb) as dA, D.alloc(n, n, nb) as dB, D.alloc(n, n, nb) as dX:
        for src, dst, w in ((hA, dA, wide[0]), (hB, dB, wide[1]), (hB, dX, wide[2])):
            resident(ch, seq, src, dst, w)
        ch.check(ch.lib.CHAMELEON_dposv_Tile_Async(LOWER, dA.ptr, dB.ptr, seq.ptr, seq.req))
        ch.check(ch.lib.CHAMELEON_dpotrs_Tile_Async(LOWER, dA.ptr, dX.ptr, seq.ptr, seq.req))
        ch.check(seq.wait())
        assert oracle.rel_frobenius(dB.to_array(n, n), want) <= 1e-12
        assert oracle.rel_frobenius(dX.to_array(n, n), want) <= 1e-12
    seq.destroy()
