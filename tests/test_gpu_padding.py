"""Device mirrors whose padding changes between operations.

A copy (dlacpy) leaves zeros on the padded diagonal, a factorisation wants ones
there.  Sizes: full tiles and an even end (nothing padded), a last tile one
short of, at and past a multiple of 16, tiles that are no multiple of 16 (all
padded), one partial tile, right-hand sides that end inside a tile.  The solve of
a copied matrix against numpy in FP64: cond(A) is O(1) for these matrices, so
the relative error is a few n eps, 1e-12 at most.
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

LOWER, FULL = 122, 123


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.init()
    yield ch


@pytest.mark.parametrize("n,nb,nrhs", [(256, 64, 64), (255, 64, 3), (257, 64, 65), (240, 64, 16), (150, 50, 7),
                                       (97, 128, 1), (600, 200, 20), (640, 320, 33)])
def test_solve_of_a_copy(ch, n, nb, nrhs):
    print("[case] padding", n, nb, nrhs, flush=True)
    L = ch.lib
    A = oracle.dplgsy(float(n), FULL, n, 3)
    B = oracle.dplrnt(n, nrhs, 4)
    want = np.linalg.solve(A, B)
    seq = ch.Sequence()
    with ch.Desc.from_array(A.copy(order="F"), nb) as dA0, ch.Desc.from_array(B.copy(order="F"), nb) as dB0, \
            ch.Desc.alloc(n, n, nb) as dA, ch.Desc.alloc(n, nrhs, nb) as dX:
        for _ in range(2):       # the second time the copy's target holds a factor
            ch.check(L.CHAMELEON_dlacpy_Tile_Async(FULL, dA0.ptr, dA.ptr, seq.ptr, seq.req))
            ch.check(L.CHAMELEON_dlacpy_Tile_Async(FULL, dB0.ptr, dX.ptr, seq.ptr, seq.req))
            ch.check(L.CHAMELEON_dposv_Tile_Async(LOWER, dA.ptr, dX.ptr, seq.ptr, seq.req))
            ch.check(seq.wait())
            X = dX.to_array(n, nrhs)
            assert oracle.rel_frobenius(X, want) <= 1e-12
    seq.destroy()
