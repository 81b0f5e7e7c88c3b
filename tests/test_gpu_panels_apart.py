"""Reduced-precision solves with the panel factored by separate launches.

CHAMAMD_PANEL=0: POTRF and TRSM apart, the panel lowered by a launch of its own
(64 x 64 blocks turned in LDS for the BF16 planes).  One, two and four 128 blocks
a tile, with a ragged last tile.  The refinement has to converge to the FP64
solution, in as many steps as the products' precision takes: forward error
against numpy 1e-12 at most, cond(A) = O(1).
"""
import ctypes
import os

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

LOWER, FULL = 122, 123
FP32, BF16, BF16X3, ADAPTIVE = 0, 1, 2, 4
STEPS = {FP32: 3, BF16: 12, BF16X3: 4, ADAPTIVE: 8}


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.finalize()
    os.environ["CHAMAMD_PANEL"] = "0"
    ch.init()
    yield ch
    ch.finalize()
    del os.environ["CHAMAMD_PANEL"]
    ch.init()


@pytest.mark.parametrize("n,nb", [(700, 128), (1100, 256), (1700, 512)])
@pytest.mark.parametrize("prec", [FP32, BF16, BF16X3, ADAPTIVE])
def test_refined_solve(ch, n, nb, prec):
    print("[case] panels apart", n, nb, prec, flush=True)
    A = oracle.dplgsy(float(n), FULL, n, 3)
    B = oracle.dplrnt(n, 2, 4)
    want = np.linalg.solve(A, B)
    it, berr = ctypes.c_int(), ctypes.c_double()
    seq = ch.Sequence()
    with ch.Desc.from_array(A.copy(order="F"), nb) as dA, ch.Desc.from_array(B.copy(order="F"), nb) as dB, \
            ch.Desc.alloc(n, 2, nb) as dX:
        ch.check(ch.lib.CHAMAMD_dposv_mixed_Tile_Async(LOWER, dA.ptr, dB.ptr, dX.ptr, prec, ctypes.byref(it),
                                                       ctypes.byref(berr), seq.ptr, seq.req))
        assert seq.wait() == 0
        X = dX.to_array(n, 2)
    seq.destroy()
    assert 0 <= it.value <= STEPS[prec], it.value
    assert oracle.rel_frobenius(X, want) <= 1e-12
