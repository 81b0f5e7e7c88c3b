"""Transfers through the staging chunks after a call that streamed its factor."""
import ctypes

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


def test_transfers_after_a_streamed_factor(ch):
    """A LAPACK-layout factorisation downloads on a stream that ends with the
    call; the staging chunks' next users must not wait on that stream."""
    n, nb, nrhs = 700, 128, 3
    A = oracle.dplgsy(float(n), FULL, n, 3)
    B = oracle.dplrnt(n, nrhs, 4)
    want = np.linalg.solve(A, B)
    ch.set_param(ch.TILE_SIZE, nb)
    for _ in range(4):
        F, X = A.copy(order="F"), B.copy(order="F")
        p = [M.ctypes.data_as(ctypes.c_void_p) for M in (F, X)]
        assert ch.lib.CHAMELEON_dposv(LOWER, n, nrhs, p[0], n, p[1], n) == 0
        assert oracle.rel_frobenius(X, want) <= 1e-12
        for m in (64, 300):
            with ch.Desc.from_array(B[:m].copy(order="F"), 64) as d:
                ch.lib.CHAMELEON_Desc_Acquire(d.ptr)
                assert (d.to_array(m, nrhs) == B[:m]).all()
