"""Reduced-precision trailing products where a wrong one cannot pass.

A has a spectrum from 1 to 1e-3 in random directions, so that the trailing
products are as large as what they are taken from, and the count of refinement
steps says whether the factor has the precision of its products.  In numpy (the
same blocked factorisation with the operands rounded, FP32 sums), corrections:
  FP32 2, BF16 8 to 11, split BF16 3; split BF16 without one of its low planes
  8 to 11; products left out, of the wrong sign, of the first panel only or
  with one tile missing: no convergence;
with the off-diagonal tiles scaled by 0.4 per tile of distance and per-tile
precision at 1e-3 (FP64, FP32 and BF16 tiles in one factorisation) 2; with 1100 rows
and more, without the
BF16 products 7, without the FP32 ones 12.
The limits below lie between.  Forward error: cond(A) 1e-13.  Each with the fused
panel, which stores the lower precision itself, and with CHAMAMD_PANEL=0, where a
launch of its own does.
"""
import ctypes
import functools
import os

import numpy as np
import pytest
from scipy.fft import dct

import oracle

pytestmark = pytest.mark.gpu

LOWER, UPPER = 122, 121
FP32, BF16, BF16X3, ADAPTIVE = 0, 1, 2, 4
LIMIT = {FP32: 3, BF16: 15, BF16X3: 5, ADAPTIVE: 3}
KAPPA = 1e3


@pytest.fixture(scope="module", params=["fused", "apart"])
def ch(request):
    import chameleon_amd as ch
    if request.param == "apart":
        ch.finalize()
        os.environ["CHAMAMD_PANEL"] = "0"
    ch.init()
    ch.panels = request.param
    yield ch
    if request.param == "apart":
        ch.finalize()
        del os.environ["CHAMAMD_PANEL"]
        ch.init()


@functools.lru_cache(maxsize=2)
def system(n, nb):
    """Q diag(lambda) Q^T with Q from two cosine transforms and random signs; nb: tiles scaled apart."""
    rng = np.random.default_rng(n)
    A = np.diag(KAPPA ** (-np.arange(n) / (n - 1.0)))
    for _ in range(2):
        s = rng.choice((-1.0, 1.0), n)
        A = dct(dct(s[:, None] * A * s, axis=0, norm="ortho"), axis=1, norm="ortho")
    A = (A + A.T) / 2
    if nb:
        t = np.arange(n) // nb
        A = A * 0.4 ** np.abs(t[:, None] - t)
    B = rng.uniform(-0.5, 0.5, (n, 2))
    return np.asfortranarray(A), np.asfortranarray(B), np.linalg.solve(A, B)


@pytest.mark.parametrize("prec", [FP32, BF16, BF16X3, ADAPTIVE])
@pytest.mark.parametrize("n,nb,uplo", [(300, 128, LOWER), (700, 384, LOWER), (1100, 128, LOWER), (2500, 256, UPPER),
                                       (3000, 512, LOWER), (5500, 128, LOWER)])
def test_refinement_steps(ch, n, nb, uplo, prec):
    print("[case] lp products", ch.panels, n, nb, uplo, prec, flush=True)
    A, B, want = system(n, nb if prec == ADAPTIVE else 0)
    it, berr = ctypes.c_int(), ctypes.c_double()
    seq = ch.Sequence()
    assert ch.lib.CHAMAMD_Set_Tile_Accuracy(ctypes.c_double(1e-3)) == 0
    try:
        with ch.Desc.from_array(A.copy(order="F"), nb) as dA, ch.Desc.from_array(B.copy(order="F"), nb) as dB, \
                ch.Desc.alloc(n, 2, nb) as dX:
            ch.check(ch.lib.CHAMAMD_dposv_mixed_Tile_Async(uplo, dA.ptr, dB.ptr, dX.ptr, prec, ctypes.byref(it),
                                                           ctypes.byref(berr), seq.ptr, seq.req))
            assert seq.wait() == 0
            X = dX.to_array(n, 2)
    finally:
        ch.lib.CHAMAMD_Set_Tile_Accuracy(ctypes.c_double(1e-12))
    seq.destroy()
    assert 0 <= it.value <= LIMIT[prec], it.value
    assert oracle.rel_frobenius(X, want) <= KAPPA * 1e-13
