"""Trailing updates whose launches cross the lines between block sizes.

The block size of a trailing update follows the number of 64 x 64 blocks in the
launch: factorisations with many and few tiles, tile sizes that are odd
multiples of 32 x 32, 64 x 64 and 128 x 128 blocks, one step and paired steps,
so that each size of block takes whole triangles and lookahead columns.  The
factor against the matrix it came from: |A - L L^T| / |A| <= n eps, the usual
bound of the factorisation with room of a factor of several.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LOWER, UPPER, FULL = 122, 121, 123


@pytest.fixture(scope="module")
def ch():
    import chameleon_amd as ch
    ch.init()
    yield ch


@pytest.mark.parametrize("n,nb,uplo", [(192, 64, LOWER), (640, 64, LOWER), (1000, 64, UPPER), (1536, 192, LOWER),
                                       (1920, 128, LOWER), (2560, 320, LOWER), (4000, 320, UPPER),
                                       (5120, 128, LOWER), (6144, 512, LOWER), (8192, 256, UPPER),
                                       (13312, 128, LOWER)])
def test_factor(ch, n, nb, uplo):
    print("[case] update", n, nb, uplo, flush=True)
    rng = np.random.default_rng(n + nb)
    A = rng.uniform(-0.5, 0.5, (n, n))
    A = np.asfortranarray(A + A.T)
    A[np.diag_indices(n)] += float(n)
    seq = ch.Sequence()
    with ch.Desc.from_array(A.copy(order="F"), nb) as dA:
        ch.check(ch.lib.CHAMELEON_dpotrf_Tile_Async(uplo, dA.ptr, seq.ptr, seq.req))
        assert seq.wait() == 0
        F = dA.to_array(n, n)
    seq.destroy()
    G = torch.from_numpy(F).cuda()
    G = G.tril() if uplo == LOWER else G.triu()
    D = torch.from_numpy(A).cuda()
    P = G @ G.T if uplo == LOWER else G.T @ G
    assert float((P - D).norm() / D.norm()) <= n * np.finfo(float).eps


SMALL_COLS = """
import sys
import numpy as np
import chameleon_amd as ch
ch.init()
n, nb = 2560, 256
rng = np.random.default_rng(3)
A = rng.uniform(-0.5, 0.5, (n, n))
A = np.asfortranarray(A + A.T)
A[np.diag_indices(n)] += float(n)
seq = ch.Sequence()
with ch.Desc.from_array(A, nb) as dA:
    ch.check(ch.lib.CHAMELEON_dpotrf_Tile_Async(122, dA.ptr, seq.ptr, seq.req))
    assert seq.wait() == 0
    np.save(sys.argv[1], dA.to_array(n, n))
"""


def test_column_blocks_switch(tmp_path):
    """CHAMAMD_SMALL_COLS=0 (large blocks in the lookahead columns, read once per
    process): the same sums, so the same bits."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = []
    for v in ("1", "0"):
        path = str(tmp_path / ("factor%s.npy" % v))
        env = dict(os.environ, CHAMAMD_SMALL_COLS=v, PYTHONPATH=root)
        subprocess.run([sys.executable, "-c", SMALL_COLS, path], check=True, env=env, timeout=100)
        out.append(np.load(path))
    assert np.array_equal(out[0], out[1])
