"""Reduced-precision trailing updates at the sizes where their blocks change.

Refined solves with FP32, BF16 and split-BF16 products and with the per-tile
precision map: few and many tiles, tile sizes of one, two and four 128 blocks,
so that 32, 64 and 128 blocks take lookahead columns and whole triangles.  The
refinement has to converge (ITER >= 0) to the FP64 solution: forward error
against numpy of a few n eps for cond(A) = O(1), 1e-12 at most.  The iteration
count says whether the factor has the precision of its products.
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

LOWER, UPPER, FULL = 122, 121, 123
FP32, BF16, BF16X3, ADAPTIVE = 0, 1, 2, 4
STEPS = {FP32: 3, BF16: 12, BF16X3: 4, ADAPTIVE: 8}


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.init()
    yield ch


@pytest.mark.parametrize("n,nb", [(300, 128), (1100, 128), (2500, 256), (3000, 512), (5500, 128)])
@pytest.mark.parametrize("prec", [FP32, BF16, BF16X3, ADAPTIVE])
def test_refined_solve(ch, n, nb, prec):
    print("[case] lp update", n, nb, prec, flush=True)
    A = oracle.dplgsy(float(n), FULL, n, 3)
    B = oracle.dplrnt(n, 2, 4)
    want = np.linalg.solve(A, B)
    it, berr = ctypes.c_int(), ctypes.c_double()
    seq = ch.Sequence()
    uplo = UPPER if n == 2500 else LOWER
    with ch.Desc.from_array(A.copy(order="F"), nb) as dA, ch.Desc.from_array(B.copy(order="F"), nb) as dB, \
            ch.Desc.alloc(n, 2, nb) as dX:
        ch.check(ch.lib.CHAMAMD_dposv_mixed_Tile_Async(uplo, dA.ptr, dB.ptr, dX.ptr, prec, ctypes.byref(it),
                                                       ctypes.byref(berr), seq.ptr, seq.req))
        assert seq.wait() == 0
        X = dX.to_array(n, 2)
    seq.destroy()
    assert 0 <= it.value <= STEPS[prec], it.value
    assert oracle.rel_frobenius(X, want) <= 1e-12
