"""Triangular solves over the widths and lengths at which their chunks change.

Right-hand sides in chunks of 16 or 32 columns, one or several launches, an odd
number of strips, the lengths just at and past the line between the two; a
solve after a factorisation that failed.  Solutions by their residual:
|A X - B| / (n max|A| max|X|) is a small multiple of eps (n eps bounds the
rounding of a backward stable solve and of the product that checks it).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LOWER, UPPER = 122, 121


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.init()
    yield ch


def matrix(n, seed):
    A = np.random.default_rng(seed).uniform(-0.5, 0.5, (n, n))
    A = np.asfortranarray(A + A.T)
    A[np.diag_indices(n)] += float(n)
    return A


def check(A, X, B):
    a, x, b = (torch.from_numpy(np.ascontiguousarray(m)).cuda() for m in (A, X, B))
    n = A.shape[0]
    r = float((a @ x - b).abs().max())
    assert r <= 4 * np.finfo(float).eps * n * float(a.abs().max()) * float(x.abs().max())


SHORT = [(64, 64, (9, 16, 17, 33)), (640, 128, (9, 16, 30, 32, 48, 64, 65, 100, 128, 150)),
         (1000, 192, (31, 47, 63, 96, 112)), (4096, 320, (16, 48, 64, 130))]
LONG = [(12288, 256, (64, 32)), (12353, 64, (64, 48, 80)), (25000, 512, (32,))]


@pytest.mark.parametrize("n,nb,widths,uplo", [c + (u,) for c in SHORT for u in (LOWER, UPPER)] +
                         [c + (LOWER,) for c in LONG])
def test_widths(ch, n, nb, widths, uplo):
    A = matrix(n, n)
    seq = ch.Sequence()
    with ch.Desc.from_array(A.copy(order="F"), nb) as dA:
        ch.check(ch.lib.CHAMELEON_dpotrf_Tile_Async(uplo, dA.ptr, seq.ptr, seq.req))
        assert seq.wait() == 0
        for k in widths:
            print("[case] strips", n, nb, k, uplo, flush=True)
            B = np.asfortranarray(np.random.default_rng(k).standard_normal((n, k)))
            with ch.Desc.from_array(B.copy(order="F"), nb) as dB:
                for _ in range(2):       # the second solves the first's solution
                    ch.check(ch.lib.CHAMELEON_dpotrs_Tile_Async(uplo, dA.ptr, dB.ptr, seq.ptr, seq.req))
                    assert seq.wait() == 0
                    X = dB.to_array(n, k)
                    check(A, X, B)
                    B = X
    seq.destroy()


@pytest.mark.parametrize("k", [1, 20])
def test_solve_after_a_failed_factorisation(ch, k):
    n, nb = 700, 128
    A = matrix(n, 5)
    bad = A.copy(order="F")
    bad[300, 300] = -1.0
    B = np.asfortranarray(np.random.default_rng(k).standard_normal((n, k)))
    for _ in range(2):
        for M, info in ((bad, 301), (A, 0)):
            seq = ch.Sequence()
            with ch.Desc.from_array(M.copy(order="F"), nb) as dA, ch.Desc.from_array(B.copy(order="F"), nb) as dB:
                ch.lib.CHAMELEON_dposv_Tile_Async(LOWER, dA.ptr, dB.ptr, seq.ptr, seq.req)
                assert seq.wait() == info
                if info == 0:
                    check(A, dB.to_array(n, k), B)
            seq.destroy()


@pytest.mark.parametrize("n,nb,k", [(1408, 128, 1), (1500, 128, 2), (1537, 128, 1), (2000, 384, 2), (4100, 256, 1),
                                    (4100, 256, 2), (4100, 256, 3), (9000, 512, 1)])
@pytest.mark.parametrize("uplo", [LOWER, UPPER])
def test_few_columns(ch, n, nb, k, uplo):
    """One to three columns about the lines between the narrow solve with its
    predecessor products and the 16-column chunks."""
    print("[case] few columns", n, nb, k, uplo, flush=True)
    A = matrix(n, n)
    B = np.asfortranarray(np.random.default_rng(k).standard_normal((n, k)))
    seq = ch.Sequence()
    with ch.Desc.from_array(A.copy(order="F"), nb) as dA, ch.Desc.from_array(B.copy(order="F"), nb) as dB, \
            ch.Desc.from_array(B.copy(order="F"), nb) as dX:
        ch.check(ch.lib.CHAMELEON_dposv_Tile_Async(uplo, dA.ptr, dB.ptr, seq.ptr, seq.req))
        ch.check(ch.lib.CHAMELEON_dpotrs_Tile_Async(uplo, dA.ptr, dX.ptr, seq.ptr, seq.req))
        assert seq.wait() == 0
        check(A, dB.to_array(n, k), B)
        check(A, dX.to_array(n, k), B)
    seq.destroy()
