"""Tiles whose columns reach past 2^31 bytes.

Two tiles of 16400 (padded to 16448) and of 16512 rows: the second tile row of the
first panel is addressed over the whole width of a tile.  The backward error
max |B - A X| / (|A| |X| N eps) of a backward stable solve is of the order of one
at most; the refined solve's test asks for |R| <= |X| |A| eps sqrt(N), so at most
1 / sqrt(N).
"""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

LOWER, UPPER, FULL = 122, 121, 123


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.init()
    ch.lib.CHAMAMD_Backward_Error.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                                              ctypes.POINTER(ctypes.c_double)]
    yield ch


def system(ch, seq, n, nb, nrhs):
    A, B, X = ch.Desc.alloc(n, n, nb), ch.Desc.alloc(n, nrhs, nb), ch.Desc.alloc(n, nrhs, nb)
    ch.check(ch.lib.CHAMELEON_dplgsy_Tile_Async(ctypes.c_double(n), FULL, A.ptr, 3, seq.ptr, seq.req))
    ch.check(ch.lib.CHAMELEON_dplrnt_Tile_Async(B.ptr, 4, seq.ptr, seq.req))
    return A, B, X


@pytest.mark.parametrize("n,nb,nrhs,uplo", [(16500, 16400, 3, LOWER), (16600, 16512, 1, LOWER)])
def test_dposv(ch, n, nb, nrhs, uplo):
    print("[case] large tiles", n, nb, nrhs, uplo, flush=True)
    seq = ch.Sequence()
    be = ctypes.c_double()
    A, B, X = system(ch, seq, n, nb, nrhs)
    with A, B, X, ch.Desc.alloc(n, n, nb) as F:
        ch.check(ch.lib.CHAMELEON_dlacpy_Tile_Async(FULL, A.ptr, F.ptr, seq.ptr, seq.req))
        ch.check(ch.lib.CHAMELEON_dlacpy_Tile_Async(FULL, B.ptr, X.ptr, seq.ptr, seq.req))
        ch.check(ch.lib.CHAMELEON_dposv_Tile_Async(uplo, F.ptr, X.ptr, seq.ptr, seq.req))
        assert seq.wait() == 0
        assert ch.lib.CHAMAMD_Backward_Error(uplo, A.ptr, X.ptr, B.ptr, ctypes.byref(be)) == 0
    seq.destroy()
    assert 0.0 <= be.value <= 1.0


@pytest.mark.parametrize("prec", [0, 2])
def test_refined(ch, prec):
    n, nb, nrhs = 16600, 16512, 1
    print("[case] large tiles, refined", prec, flush=True)
    seq = ch.Sequence()
    it, berr, be = ctypes.c_int(), ctypes.c_double(), ctypes.c_double()
    A, B, X = system(ch, seq, n, nb, nrhs)
    with A, B, X:
        ch.check(ch.lib.CHAMAMD_dposv_mixed_Tile_Async(LOWER, A.ptr, B.ptr, X.ptr, prec, ctypes.byref(it),
                                                       ctypes.byref(berr), seq.ptr, seq.req))
        assert seq.wait() == 0
        assert ch.lib.CHAMAMD_Backward_Error(LOWER, A.ptr, X.ptr, B.ptr, ctypes.byref(be)) == 0
    seq.destroy()
    assert 0 <= it.value <= 5
    assert 0.0 <= be.value <= n ** -0.5
