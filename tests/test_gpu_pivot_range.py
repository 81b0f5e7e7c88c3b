"""Pivots at the ends of the range of FP64.

A = s^2 L0 L0^T with L0 lower triangular, 4 on its diagonal, 1 on three lower
ones: integers, so A is exact for every power of two s whose A is representable,
every pivot is 16 s^2 and the factor is s L0.  The inverse of L0 is bounded (rows
of 4 and at most 3), so the factor is as exact as a factorisation of L0 L0^T by
itself, 1e-13; solutions of A X = A Xi with small integers Xi likewise, 1e-12.
s^2 = 2^-1040 makes A subnormal (integers below 2^34 are exact there) and 1 / d
infinite, 2^1018 makes 1 / d subnormal.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LOWER, UPPER = 122, 121
SCALES = [-1040, -1020, 0, 1018]


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.init()
    yield ch


def matrix(n, e):
    L0 = 4.0 * np.eye(n) + sum(np.eye(n, k=-k) for k in (1, 17, 70))
    rng = np.random.default_rng(n)
    X = rng.integers(-3, 4, (n, 3)).astype(float)
    A = np.ldexp(L0 @ L0.T, e)
    B = np.ldexp((L0 @ (L0.T @ X)), e) if e < 1000 else np.ldexp(L0 @ (L0.T @ X), 0)
    return np.asfortranarray(A), np.asfortranarray(B), L0, X if e < 1000 else np.ldexp(X, -e)


def close(a, b, tol):
    m = np.abs(b).max()
    return np.abs(a / m - b / m).max() <= tol


@pytest.mark.parametrize("e", SCALES)
@pytest.mark.parametrize("n,nb,uplo", [(16, 64, LOWER), (64, 64, LOWER), (100, 40, UPPER), (200, 128, UPPER),
                                       (333, 64, LOWER)])
def test_factor_and_solve(ch, n, nb, uplo, e):
    print("[case] pivots 2^%d" % e, n, nb, uplo, flush=True)
    A, B, L0, X = matrix(n, e)
    seq = ch.Sequence()
    with ch.Desc.from_array(A, nb) as dA, ch.Desc.from_array(B, nb) as dB:
        ch.check(ch.lib.CHAMELEON_dposv_Tile_Async(uplo, dA.ptr, dB.ptr, seq.ptr, seq.req))
        assert seq.wait() == 0
        F, Y = dA.to_array(n, n), dB.to_array(n, 3)
    seq.destroy()
    F = np.tril(F) if uplo == LOWER else np.triu(F).T
    assert close(F, np.ldexp(L0, e // 2), 1e-13)
    assert close(Y, X, 1e-12)


@pytest.mark.parametrize("last", [0, 15, 16, 40, 63, 64, 99])
def test_one_tiny_pivot(ch, last):
    """One pivot far below the others, first, last and in between."""
    n, nb = 100, 100
    print("[case] one tiny pivot", last, flush=True)
    d = np.full(n, 4.0)
    d[last] = 2.0 ** -1040
    A = np.asfortranarray(np.diag(d))
    seq = ch.Sequence()
    with ch.Desc.from_array(A, nb) as dA:
        ch.lib.CHAMELEON_dpotrf_Tile_Async(LOWER, dA.ptr, seq.ptr, seq.req)
        assert seq.wait() == 0
        F = np.tril(dA.to_array(n, n))
    seq.destroy()
    assert np.abs(F / np.sqrt(np.diag(d)).max(axis=0) - np.eye(n)).max() <= 1e-15


@pytest.mark.parametrize("n,nb,uplo", [(60, 64, LOWER), (150, 64, UPPER), (300, 200, LOWER)])
def test_rows_of_every_scale(ch, n, nb, uplo):
    """D L0 L0^T D with powers of two from 2^-512 to 2^507 in D: both ends of the range in one
    16-column step, each row as exact as without D."""
    print("[case] rows of every scale", n, nb, uplo, flush=True)
    _, _, L0, _ = matrix(n, 0)
    rng = np.random.default_rng(2 * n)
    k = rng.integers(-512, 508, n)
    k[[3, 9]] = 507, -512
    X = rng.integers(-3, 4, (n, 2)).astype(float)
    A = np.asfortranarray(np.ldexp(L0 @ L0.T, k[:, None] + k))
    B = np.asfortranarray(np.ldexp(L0 @ (L0.T @ X), k[:, None]))
    seq = ch.Sequence()
    with ch.Desc.from_array(A, nb) as dA, ch.Desc.from_array(B, nb) as dB:
        ch.check(ch.lib.CHAMELEON_dposv_Tile_Async(uplo, dA.ptr, dB.ptr, seq.ptr, seq.req))
        assert seq.wait() == 0
        F, Y = dA.to_array(n, n), dB.to_array(n, 2)
    seq.destroy()
    F = np.tril(F) if uplo == LOWER else np.triu(F).T
    assert np.abs(np.ldexp(F, -k[:, None]) - L0).max() <= 4.0 * 1e-13
    assert np.abs(np.ldexp(Y, k[:, None]) - X).max() <= 3.0 * 1e-12


def test_not_positive_after_a_tiny_pivot(ch):
    n, nb = 100, 100
    d = np.full(n, 2.0 ** -1040)
    d[70] = -d[70]
    seq = ch.Sequence()
    with ch.Desc.from_array(np.asfortranarray(np.diag(d)), nb) as dA:
        ch.lib.CHAMELEON_dpotrf_Tile_Async(LOWER, dA.ptr, seq.ptr, seq.req)
        assert seq.wait() == 71
    seq.destroy()


@pytest.mark.parametrize("e", SCALES)
def test_batch(ch, e):
    sizes = [1, 16, 40, 64, 100, 333]
    print("[case] batched pivots 2^%d" % e, flush=True)
    n = np.array(sizes, dtype=np.int32)
    k = np.full(len(n), 3, dtype=np.int32)
    ip = ctypes.POINTER(ctypes.c_int)
    info = np.zeros(len(n), dtype=np.int32)
    b = ctypes.c_void_p()
    L = ch.lib
    ch.check(L.CHAMAMD_Batch_Create(ctypes.byref(b), len(n), n.ctypes.data_as(ip), k.ctypes.data_as(ip)))
    want = []
    for i, m in enumerate(sizes):
        A, B, _, X = matrix(m, e)
        want.append(X)
        ch.check(L.CHAMAMD_Batch_SetA(b, i, LOWER, ctypes.c_void_p(A.ctypes.data), m))
        ch.check(L.CHAMAMD_Batch_SetB(b, i, ctypes.c_void_p(B.ctypes.data), m))
    ch.check(L.CHAMAMD_dposv_batch(b, info.ctypes.data_as(ip)))
    got = []
    for i, m in enumerate(sizes):
        Y = np.zeros((m, 3), order="F")
        ch.check(L.CHAMAMD_Batch_GetB(b, i, ctypes.c_void_p(Y.ctypes.data), m))
        got.append(Y)
    L.CHAMAMD_Batch_Destroy(ctypes.byref(b))
    assert not info.any()
    for Y, X in zip(got, want):
        assert close(Y, X, 1e-12)
