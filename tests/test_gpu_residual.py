"""FP64 residual, its column maxima and the norm of the working copy at the sizes
where their launches change: one column group, whole 64-column chunks and
ragged column counts, 8 to 32 pieces of the row range, tiles of one to eight
128-row groups cut in one or more column pieces.

The backward error of integer matrices is exact: every product and sum is
a small integer, so residual, norms and maxima have one value each and
only the final quotient rounds (1e-14).  The norm that the mixed solve forms
with its copy differs from the plain norm by the order of its sums: N eps, 1e-12.
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
    ch.lib.CHAMAMD_Backward_Error.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                                              ctypes.POINTER(ctypes.c_double)]
    yield ch


@pytest.mark.parametrize("uplo", [LOWER, UPPER])
@pytest.mark.parametrize("n,nb,nrhs", [(5, 32, 1), (130, 64, 16), (300, 100, 17), (700, 128, 40), (700, 320, 64),
                                       (1500, 96, 100), (2600, 512, 130), (9000, 256, 2), (17000, 512, 1)])
def test_backward_error_exact(ch, uplo, n, nb, nrhs):
    print("[case] residual", uplo, n, nb, nrhs, flush=True)
    rng = np.random.default_rng(n + nrhs)
    A = np.asfortranarray(rng.integers(-9, 10, (n, n)).astype(float))
    S = np.tril(A) + np.tril(A, -1).T if uplo == LOWER else np.triu(A) + np.triu(A, 1).T
    X = np.asfortranarray(rng.integers(-9, 10, (n, nrhs)).astype(float))
    B = np.asfortranarray(rng.integers(-99, 100, (n, nrhs)).astype(float))
    R = np.abs(B - S @ X).max(axis=0)
    want = (R / (np.abs(S).sum(axis=1).max() * np.abs(X).max(axis=0) * n * 2.0 ** -53)).max()
    be = ctypes.c_double()
    with ch.Desc.from_array(A, nb) as dA, ch.Desc.from_array(X, nb) as dX, ch.Desc.from_array(B, nb) as dB:
        assert ch.lib.CHAMAMD_Backward_Error(uplo, dA.ptr, dX.ptr, dB.ptr, ctypes.byref(be)) == 0
    assert abs(be.value - want) <= 1e-14 * want, (be.value, want)


@pytest.mark.parametrize("n,nb,nrhs", [(128, 128, 1), (900, 384, 3), (1300, 640, 20), (2100, 1024, 64), (1030, 256, 2),
                                       (6000, 128, 1)])
def test_copy_norm(ch, n, nb, nrhs):
    print("[case] copy norm", n, nb, nrhs, flush=True)
    A = oracle.dplgsy(float(n), FULL, n, 7)
    A[0, 1:] *= 3.0     # the longest row sum is the first one
    A[1:, 0] *= 3.0
    B = oracle.dplrnt(n, nrhs, 8)
    want = np.linalg.solve(A, B)
    it, be, ref = ctypes.c_int(), ctypes.c_double(), ctypes.c_double()
    seq = ch.Sequence()
    with ch.Desc.from_array(A.copy(order="F"), nb) as dA, ch.Desc.from_array(B.copy(order="F"), nb) as dB, \
            ch.Desc.alloc(n, nrhs, nb) as dX:
        ch.check(ch.lib.CHAMAMD_dposv_mixed_Tile_Async(LOWER, dA.ptr, dB.ptr, dX.ptr, 0, ctypes.byref(it),
                                                       ctypes.byref(be), seq.ptr, seq.req))
        assert seq.wait() == 0
        assert ch.lib.CHAMAMD_Backward_Error(LOWER, dA.ptr, dX.ptr, dB.ptr, ctypes.byref(ref)) == 0
        X = dX.to_array(n, nrhs)
    seq.destroy()
    assert 0 <= it.value <= 3
    assert abs(be.value - ref.value) <= 1e-12 * ref.value, (be.value, ref.value)
    assert oracle.rel_frobenius(X, want) <= 1e-12


@pytest.mark.parametrize("n,nb,nrhs", [(1152, 1152, 1), (2500, 1152, 5), (1400, 1408, 2), (3000, 1408, 1),
                                       (1664, 1664, 1), (4000, 1920, 17)])
def test_copy_norm_odd_multiples_of_128(ch, n, nb, nrhs):
    """Tiles whose column pieces stop at an odd multiple of eight columns."""
    test_copy_norm(ch, n, nb, nrhs)


@pytest.mark.parametrize("n,nb,nrhs", [(1500, 512, 1), (1700, 384, 2), (3500, 512, 1)])
def test_narrow_solve_behind_odd_tile_counts(ch, n, nb, nrhs):
    """The strip inverses of one or two columns come after NT^2 tile norms, an odd
    number of doubles here; the launch checks that they are on 32 bytes."""
    test_copy_norm(ch, n, nb, nrhs)
