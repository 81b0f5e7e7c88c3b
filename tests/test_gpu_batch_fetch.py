"""Right-hand sides fetched from a batch: one by one, in runs, and out of order.

Runs of calls read ahead, so the values must be those of the moment of the call
whatever changed B in between: the fetched values equal the ones that were set
(bit for bit), or the generated ones (one column each, against the oracle).
"""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.init()
    yield ch


@pytest.mark.parametrize("count,hi,nrhs_hi", [(1, 40, 3), (15, 40, 3), (17, 40, 1), (31, 70, 4), (33, 70, 4), (200, 90, 5),
                                              (70, 2000, 140)])
def test_fetch_in_any_order(ch, count, hi, nrhs_hi):
    print("[case] fetch", count, hi, nrhs_hi, flush=True)
    rng = np.random.default_rng(count)
    n = rng.integers(1, hi, count).astype(np.int32)
    nrhs = rng.integers(0, nrhs_hi + 1, count).astype(np.int32)
    if count == 70:
        n[40], nrhs[40] = 2000, 600                          # larger than the read-ahead buffer
    ip = ctypes.POINTER(ctypes.c_int)
    b = ctypes.c_void_p()
    L = ch.lib
    ch.check(L.CHAMAMD_Batch_Create(ctypes.byref(b), count, n.ctypes.data_as(ip), nrhs.ctypes.data_as(ip)))
    B = [np.asfortranarray(rng.standard_normal((n[i], nrhs[i]))) for i in range(count)]

    def put(i):
        ch.check(L.CHAMAMD_Batch_SetB(b, i, _p(B[i]), int(n[i])))

    def same(i, pad=0):
        X = np.full((n[i] + pad, nrhs[i]), np.nan, order="F")
        ch.check(L.CHAMAMD_Batch_GetB(b, i, _p(X), int(n[i]) + pad))
        assert (X[:n[i]] == B[i]).all() and np.isnan(X[n[i]:]).all(), i

    for i in range(count):
        put(i)
    for i in range(count):
        same(i, i % 3)
    for i in range(count):                                   # again, with changes just ahead of the run
        same(i)
        if i % 9 == 5 and i + 1 < count:
            B[i + 1] = np.asfortranarray(-2.0 * B[i + 1])
            put(i + 1)
    for i in rng.integers(0, count, 3 * count):
        same(int(i))
    for i in range(count):                                   # a run that jumps back and ahead
        same(i)
        if i % 25 == 24:
            same(i - 20)
    ch.check(L.CHAMAMD_dplrnt_batch(b, 77))
    for i in range(count):
        if nrhs[i]:
            X = np.empty((n[i], nrhs[i]), order="F")
            ch.check(L.CHAMAMD_Batch_GetB(b, i, _p(X), int(n[i])))
            assert (X == oracle.dplrnt(int(n[i]), int(nrhs[i]), 77 + i)).all()
    # the matrices are identities: a solve leaves B as it is
    for i in range(count):
        put(i)
        if i % 2:
            same(i)
    for i in range(count // 2):
        same(i)
    ch.check(L.CHAMAMD_dposv_batch(b, None))
    for i in range(count // 2, count):
        same(i)
    ch.check(L.CHAMAMD_Batch_Destroy(ctypes.byref(b)))


def test_fetch_takes_no_device_memory(ch):
    """The read-ahead works where the device's memory is full: none of it is taken."""
    import torch
    count = 200000                                           # tables of 2.4 MB
    n = np.ones(count, dtype=np.int32)
    ip = ctypes.POINTER(ctypes.c_int)
    b = ctypes.c_void_p()
    L = ch.lib
    ch.check(L.CHAMAMD_Batch_Create(ctypes.byref(b), count, n.ctypes.data_as(ip), n.ctypes.data_as(ip)))
    ch.check(L.CHAMAMD_dplrnt_batch(b, 5))
    x = np.empty(100)
    ch.check(L.CHAMAMD_Batch_GetB(b, 0, ctypes.c_void_p(x.ctypes.data), 1))
    free = torch.cuda.mem_get_info()[0]
    for i in range(1, 100):
        ch.check(L.CHAMAMD_Batch_GetB(b, i, ctypes.c_void_p(x.ctypes.data + 8 * i), 1))
    assert torch.cuda.mem_get_info()[0] == free
    ch.check(L.CHAMAMD_Batch_Destroy(ctypes.byref(b)))
    assert (x == [oracle.dplrnt(1, 1, 5 + i)[0, 0] for i in range(100)]).all()
