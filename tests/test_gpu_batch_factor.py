"""Factorisation of batched systems at the edges of its blocks.

Orders around the 16- and 64-column blocks, the 64 and 128 rows that one pass of
four or eight wavefronts takes, and long ones; both workgroup shapes, FP64 and
FP32 products.  Against numpy in FP64: cond(A) is O(1), so factor and solution
agree to a few n eps, 1e-12 at most; the refined solve has the same bound.
A system that is not positive definite reports the column LAPACK does and
leaves the others as they are.
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

LOWER, FULL = 122, 123
PREC_FP32 = 0
ORDERS = [1, 15, 16, 17, 32, 33, 48, 49, 63, 64, 65, 79, 80, 81, 96, 112, 127, 128, 129, 144, 160, 191, 192, 193, 208,
          255, 256, 257, 320, 321, 336, 449, 513, 640, 705, 1023, 1100]
ip = ctypes.POINTER(ctypes.c_int)


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.init()
    yield ch


class Systems:
    def __init__(self, ch, orders, nrhs):
        self.L, self.ch = ch.lib, ch
        self.n = np.asarray(orders, dtype=np.int32)
        self.k = np.full(len(orders), nrhs, dtype=np.int32)
        self.b = ctypes.c_void_p()
        ch.check(self.L.CHAMAMD_Batch_Create(ctypes.byref(self.b), len(orders), self.n.ctypes.data_as(ip),
                                             self.k.ctypes.data_as(ip)))
        self.A = [oracle.dplgsy(float(n), FULL, int(n), 11 + i) for i, n in enumerate(orders)]
        self.B = [oracle.dplrnt(int(n), nrhs, 51 + i) for i, n in enumerate(orders)]
        self.info = np.full(len(orders), -7, dtype=np.int32)

    def put(self):
        for i, n in enumerate(self.n):
            self.ch.check(self.L.CHAMAMD_Batch_SetA(self.b, i, LOWER, _p(np.asfortranarray(self.A[i])), int(n)))
            self.ch.check(self.L.CHAMAMD_Batch_SetB(self.b, i, _p(np.asfortranarray(self.B[i])), int(n)))

    def x(self, i):
        X = np.empty((self.n[i], self.k[i]), order="F")
        self.ch.check(self.L.CHAMAMD_Batch_GetB(self.b, i, _p(X), int(self.n[i])))
        return X

    def factor(self, i):
        F = np.zeros((self.n[i], self.n[i]), order="F")
        self.ch.check(self.L.CHAMAMD_Batch_GetA(self.b, i, LOWER, _p(F), int(self.n[i])))
        return np.tril(F)

    def close(self):
        self.ch.check(self.L.CHAMAMD_Batch_Destroy(ctypes.byref(self.b)))


@pytest.mark.parametrize("waves", [4, 8])
def test_factor_and_solve(ch, waves):
    old = (ctypes.c_int * 6)()
    ch.check(ch.lib.CHAMAMD_Batch_Get_Tuning(old, None, None))
    s = Systems(ch, ORDERS, 3)
    try:
        ch.check(ch.lib.CHAMAMD_Batch_Set_Tuning((ctypes.c_int * 6)(*[waves] * 6)))
        s.put()
        assert ch.lib.CHAMAMD_dposv_batch(s.b, s.info.ctypes.data_as(ip)) == 0
        for i, n in enumerate(ORDERS):
            assert s.info[i] == 0
            assert oracle.rel_frobenius(s.factor(i), np.linalg.cholesky(s.A[i])) <= 1e-12, n
            assert oracle.rel_frobenius(s.x(i), np.linalg.solve(s.A[i], s.B[i])) <= 1e-12, n
        # refined from a factor with FP32 products
        s.put()
        it = np.zeros(len(ORDERS), dtype=np.int32)
        assert ch.lib.CHAMAMD_dposv_mixed_batch(s.b, PREC_FP32, it.ctypes.data_as(ip), s.info.ctypes.data_as(ip)) == 0
        for i, n in enumerate(ORDERS):
            assert it[i] >= 0 and s.info[i] == 0
            assert oracle.rel_frobenius(s.x(i), np.linalg.solve(s.A[i], s.B[i])) <= 1e-12, n
    finally:
        ch.check(ch.lib.CHAMAMD_Batch_Set_Tuning(old))
        s.close()


def test_not_positive_definite(ch):
    cols = {1: 1, 40: 17, 64: 64, 65: 65, 130: 100, 200: 129, 257: 257, 300: 193, 700: 650}
    orders = [n for n in cols for _ in (0, 1)]               # a bad system and a good one of each order
    s = Systems(ch, orders, 1)
    for i, n in enumerate(orders):
        if i % 2 == 0:
            s.A[i][cols[n] - 1, cols[n] - 1] = -float(n)
    s.put()
    assert ch.lib.CHAMAMD_dpotrf_batch(s.b, s.info.ctypes.data_as(ip)) != 0
    for i, n in enumerate(orders):
        assert s.info[i] == (cols[n] if i % 2 == 0 else 0), (n, s.info[i])
        if i % 2:
            assert oracle.rel_frobenius(s.factor(i), np.linalg.cholesky(s.A[i])) <= 1e-12, n
    s.close()
