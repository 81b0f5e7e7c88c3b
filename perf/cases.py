"""Workloads of the Cholesky library, for timing it over its range of use.

Every case goes through the public entry points as a caller's program does:

  posv    descriptors resident on the device (the _Tile_Async calls): the
          program keeps A and B, solves on copies (dlacpy, dposv) and brings
          the solution home (Desc_Flush, Sequence_Wait); the factor stays on
          the device
  potrs   the factor is resident, new right-hand sides are solved with it
  lapack  the LAPACK-layout drop-in on column-major host arrays; factor and
          solution come back in those arrays
  mixed   reduced-precision factorisation with FP64 iterative refinement
  batch   uneven independent systems, generated on the device, factored and
          solved in one call, every solution read back
  serve   the solve server: requests of mixed sizes arrive, some reuse an
          earlier request's matrix, progress is made between arrivals

listed() and draw() give the cases, prepare() the state a program holds before
the call, run() one pass, work() what a pass cannot do without, exact() the
same results from torch in 64 bits on inputs restated here.
"""
import ctypes
import math

import numpy as np
import torch

import chameleon_amd as ch

PREC = {"fp32": 0, "bf16x3": 2}
EXACT_MOST_SYSTEMS = 1200        # about ten seconds of small factorisations


def listed():
    return [
        # one small system handed over by a LAPACK caller: latency of the whole call
        {"name": "lapack_n96", "kind": "lapack", "n": 96, "nrhs": 1, "nb": 384, "uplo": "L"},
        # a LAPACK caller's everyday size, factor and solution back on the host
        {"name": "lapack_n1500", "kind": "lapack", "n": 1500, "nrhs": 8, "nb": 384, "uplo": "L"},
        # a small resident solve inside an application's loop: a chain of short launches
        {"name": "posv_n640", "kind": "posv", "n": 640, "nrhs": 16, "nb": 128, "uplo": "L"},
        # Chameleon's CPU configuration (N=4096, NB=320, NRHS=16)
        {"name": "posv_n4096", "kind": "posv", "n": 4096, "nrhs": 16, "nb": 320, "uplo": "L"},
        # the other triangle, an order and right-hand sides that fit no tile
        {"name": "posv_upper_n7003", "kind": "posv", "n": 7003, "nrhs": 7, "nb": 256, "uplo": "U"},
        # the headline factor-and-solve
        {"name": "posv_n32768", "kind": "posv", "n": 32768, "nrhs": 64, "nb": 512, "uplo": "L"},
        # repeated solves with a resident factor: one right-hand side, and a block of them
        {"name": "potrs_n32768_nrhs1", "kind": "potrs", "n": 32768, "nrhs": 1, "nb": 512, "uplo": "L"},
        {"name": "potrs_n32768_nrhs64", "kind": "potrs", "n": 32768, "nrhs": 64, "nb": 512, "uplo": "L"},
        # mixed precision with refinement: a moderate size, and the benchmark's
        {"name": "mixed_fp32_n4096", "kind": "mixed", "n": 4096, "nrhs": 1, "nb": 256, "uplo": "L", "prec": "fp32",
         "kappa": 100.0},
        {"name": "mixed_bf16x3_n32768", "kind": "mixed", "n": 32768, "nrhs": 64, "nb": 512, "uplo": "L",
         "prec": "bf16x3", "kappa": 10000.0},
        # the uneven batch: 20 000 systems, orders log-uniform in [16, 1024), 1 to 8 right-hand sides
        {"name": "batch_20000", "kind": "batch", "count": 20000, "lo": 16, "hi": 1024, "prec": "fp64"},
        # a burst of server requests, orders log-uniform in [64, 4096), 30 % on an earlier matrix
        {"name": "serve_96", "kind": "serve", "count": 96, "lo": 64, "hi": 4096, "nb": 256},
    ]


def _log_int(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(("lapack", "posv", "posv", "posv", "potrs", "potrs", "mixed", "batch", "serve"))
    uplo = rng.choice("LLLU")
    if kind == "lapack":
        return {"kind": kind, "n": _log_int(rng, 20, 3000), "nrhs": _log_int(rng, 1, 40),
                "nb": rng.choice((128, 256, 384)), "uplo": uplo}
    if kind in ("posv", "potrs"):
        n = _log_int(rng, 100, 24000)
        sizes = [b for b in (64, 128, 192, 256, 320, 384, 512) if n <= 80 * b]
        if n <= 4000:
            sizes.append(200)            # a tile that is no multiple of 64
        return {"kind": kind, "n": n, "nrhs": _log_int(rng, 1, 130), "nb": rng.choice(sizes), "uplo": uplo}
    if kind == "mixed":
        return {"kind": kind, "n": _log_int(rng, 500, 8000), "nrhs": _log_int(rng, 1, 80),
                "nb": rng.choice((128, 256, 384, 512)), "uplo": uplo, "prec": rng.choice(("fp32", "bf16x3")),
                "kappa": 10.0 ** rng.uniform(1.0, 4.0)}
    if kind == "batch":
        return {"kind": kind, "count": _log_int(rng, 16, 4000), "lo": 16, "hi": rng.choice((96, 300, 1024)),
                "prec": rng.choice(("fp64", "fp64", "fp32"))}
    return {"kind": kind, "count": _log_int(rng, 8, 90), "lo": 64, "hi": rng.choice((512, 1024, 4096)), "nb": 256}


# --------------------------------------------------------------- inputs

LCG = (6364136223846793005, 1)
MASK = (1 << 64) - 1


def _i64(x):
    return x - (1 << 64) if x >> 63 else x


def _compose(f, g):
    """The affine map x -> f(g(x)) modulo 2^64."""
    return (f[0] * g[0]) & MASK, (f[0] * g[1] + f[1]) & MASK


def _power(f, n):
    out = (1, 0)
    while n:
        if n & 1:
            out = _compose(f, out)
        f = _compose(f, f)
        n >>= 1
    return out


def _orbit(x, f, count):
    """Rows x, f(x), f(f(x)), ... (int64 with wrap-around), `count` of them."""
    while x.shape[0] < count:
        more = min(x.shape[0], count - x.shape[0])
        x = torch.cat((x, x[:more] * _i64(f[0]) + _i64(f[1])))
        f = _compose(f, f)
    return x


def random_matrix(m, n, seed, device):
    """Entry (i, j) is state i + j*m of the generator, as 0.5 - state * 2^-64: dplrnt."""
    cols = _orbit(torch.tensor([_i64(seed)], dtype=torch.int64, device=device), _power(LCG, m), n)
    x = _orbit(cols[None, :], LCG, m)
    v = x.to(torch.float64)
    v += (x < 0).to(torch.float64) * 2.0 ** 64
    return v.mul_(-(2.0 ** -64)).add_(0.5)


def spd_matrix(n, seed, device):
    """dplgsy with bump n: the lower triangle of random_matrix mirrored, n added to the diagonal."""
    a = random_matrix(n, n, seed, device).tril_()
    a.diagonal().add_(float(n)).mul_(0.5)
    return a + a.T


def _hartley(x, dim):
    """The orthogonal, symmetric Hartley transform along `dim`."""
    f = torch.fft.fft(x, dim=dim)
    return (f.real - f.imag) / math.sqrt(x.shape[dim])


def conditioned_matrix(n, kappa, seed):
    """Q diag(kappa^(-i/(n-1))) Q^T with Q = H S H, H the Hartley transform and S random signs."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    sign = torch.randint(0, 2, (n,), generator=g, device="cuda").to(torch.float64) * 2.0 - 1.0
    a = torch.diag(torch.logspace(0.0, -math.log10(kappa), n, dtype=torch.float64, device="cuda"))
    a = _hartley(_hartley(a, 0), 1) * sign * sign[:, None]
    a = _hartley(_hartley(a, 0), 1)
    return (a + a.T).mul_(0.5)


def _systems(case):
    """Orders, right-hand sides and (serve) the request each matrix is taken from: the case's own."""
    r = np.random.RandomState(case["count"])
    n = np.floor(np.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]), case["count"]))).astype(np.int32)
    if case["kind"] == "batch":
        return n, r.randint(1, 9, case["count"]).astype(np.int32), None
    nrhs = r.choice((1, 4, 16), case["count"]).astype(np.int32)
    source = np.arange(case["count"])
    for i in range(1, case["count"]):
        if r.uniform() < 0.3:
            source[i] = source[r.randint(0, i)]
            n[i] = n[source[i]]
    return n, nrhs, source


def _seed_a(seed):
    return 1 + 3 * seed


def _seed_b(seed):
    return 2 + 5 * seed


# ---------------------------------------------------------------- state


class State:
    """What a program keeps: descriptors, a sequence, host arrays."""

    def __init__(self, case):
        self.case = case
        self.owned = []
        self.uplo = ch.UPPER if case.get("uplo") == "U" else ch.LOWER

    def own(self, x):
        self.owned.append(x)
        return x

    def __del__(self):
        for x in reversed(self.owned):
            x.destroy()


class Batch:
    def __init__(self, n, nrhs):
        self.ptr = ctypes.c_void_p()
        ip = ctypes.POINTER(ctypes.c_int)
        ch.check(ch.lib.CHAMAMD_Batch_Create(ctypes.byref(self.ptr), len(n), n.ctypes.data_as(ip),
                                             nrhs.ctypes.data_as(ip)))

    def destroy(self):
        ch.lib.CHAMAMD_Batch_Destroy(ctypes.byref(self.ptr))


def _block(flat, at, n, k):
    """The n x k column-major block of a flat array that starts at `at`."""
    return flat[at:at + n * k].reshape(k, n).T


def prepare(case, seed):
    ch.init()
    ch.set_param(ch.TILE_SIZE, case.get("nb", 256))
    st = State(case)
    kind, L = case["kind"], ch.lib
    if kind == "lapack":
        n, k = case["n"], case["nrhs"]
        st.a0 = np.asfortranarray(spd_matrix(n, _seed_a(seed), "cpu").numpy())
        st.b0 = np.asfortranarray(random_matrix(n, k, _seed_b(seed), "cpu").numpy())
        st.a, st.b = np.empty_like(st.a0, order="F"), np.empty_like(st.b0, order="F")
        return st
    if kind == "batch":
        st.n, st.nrhs, _ = _systems(case)
        st.batch = st.own(Batch(st.n, st.nrhs))
        st.seed_a, st.seed_b = _seed_a(seed), _seed_b(seed)
        st.info = np.zeros(len(st.n), dtype=np.int32)
        st.iter = np.zeros(len(st.n), dtype=np.int32)
        st.at = np.concatenate(([0], np.cumsum(st.n.astype(np.int64) * st.nrhs)))
        st.x = np.zeros(st.at[-1])
        return st
    if kind == "serve":
        st.n, st.nrhs, st.source = _systems(case)
        st.server = st.own(ch.Server(6 << 30))
        st.next_id, st.seed_a = 0, _seed_a(seed)
        st.at = np.concatenate(([0], np.cumsum(st.n.astype(np.int64) * st.nrhs)))
        st.b0 = np.concatenate([random_matrix(int(n), int(k), _seed_b(seed) + i, "cpu").numpy().ravel(order="F")
                                for i, (n, k) in enumerate(zip(st.n, st.nrhs))])
        st.x = np.empty_like(st.b0)
        return st
    n, k, nb = case["n"], case["nrhs"], case["nb"]
    st.seq = st.own(ch.Sequence())
    s = (st.seq.ptr, st.seq.req)
    st.A0 = st.own(ch.Desc.alloc(n, n, nb))
    if kind == "mixed" and n <= 8192:
        a = np.asfortranarray(conditioned_matrix(n, case["kappa"], seed).cpu().numpy())
        host = ch.Desc.from_array(a, nb)
        ch.check(L.CHAMELEON_dlacpy_Tile_Async(ch.UPPERLOWER, host.ptr, st.A0.ptr, *s))
        ch.check(st.seq.wait())
        host.destroy()
    elif kind == "mixed":
        ch.check(L.CHAMAMD_dplgsy_cond_Tile(case["kappa"], ch.DIST_NORMAL, st.A0.ptr, seed))
        ch.check(L.CHAMAMD_Cond_Cache_Release())
    else:
        ch.check(L.CHAMELEON_dplgsy_Tile_Async(float(n), ch.UPPERLOWER, st.A0.ptr, _seed_a(seed), *s))
    st.B0 = st.own(ch.Desc.alloc(n, k, nb))
    ch.check(L.CHAMELEON_dplrnt_Tile_Async(st.B0.ptr, _seed_b(seed), *s))
    st.x = np.zeros((n, k), order="F")
    st.B = st.own(ch.Desc.from_array(st.x, nb))
    if kind == "posv":
        st.A = st.own(ch.Desc.alloc(n, n, nb))
        ch.check(L.CHAMELEON_dlacpy_Tile_Async(ch.UPPERLOWER, st.A0.ptr, st.A.ptr, *s))
    if kind == "potrs":
        ch.check(L.CHAMELEON_dpotrf_Tile_Async(st.uplo, st.A0.ptr, *s))
    ch.check(st.seq.wait())
    return st


def run(st):
    case, L = st.case, ch.lib
    kind = case["kind"]
    ip = ctypes.POINTER(ctypes.c_int)
    if kind == "lapack":
        ch.set_param(ch.TILE_SIZE, case["nb"])
        np.copyto(st.a, st.a0)
        np.copyto(st.b, st.b0)
        n = case["n"]
        ch.check(L.CHAMELEON_dposv(st.uplo, n, case["nrhs"], st.a.ctypes.data, n, st.b.ctypes.data, n))
        return {"a": st.a, "x": st.b}
    if kind == "batch":
        b = st.batch.ptr
        ch.check(L.CHAMAMD_dplgsy_batch(b, st.seed_a))
        ch.check(L.CHAMAMD_dplrnt_batch(b, st.seed_b))
        info = st.info.ctypes.data_as(ip)
        if case["prec"] == "fp64":
            ch.check(L.CHAMAMD_dposv_batch(b, info))
        else:
            ch.check(L.CHAMAMD_dposv_mixed_batch(b, PREC[case["prec"]], st.iter.ctypes.data_as(ip), info))
        x = st.x.ctypes.data
        for i, (at, n) in enumerate(zip(st.at.tolist(), st.n.tolist())):
            L.CHAMAMD_Batch_GetB(b, i, x + 8 * at, n)
        return {"x": st.x, "info": st.info}
    if kind == "serve":
        ch.set_param(ch.TILE_SIZE, case["nb"])
        np.copyto(st.x, st.b0)
        first = st.next_id
        st.next_id += case["count"]
        for i, (n, k, src) in enumerate(zip(st.n.tolist(), st.nrhs.tolist(), st.source.tolist())):
            st.server.submit(first + src, n, _block(st.x, st.at[i], n, k), seed=st.seed_a + src)
            st.server.progress()
        st.server.drain()
        done = st.server.finished()
        if len(done) != case["count"]:
            raise RuntimeError("%d of %d requests finished" % (len(done), case["count"]))
        return {"x": st.x}
    s = (st.seq.ptr, st.seq.req)
    if kind == "mixed":
        it, berr = ctypes.c_int(), ctypes.c_double()
        ch.check(L.CHAMAMD_dposv_mixed_Tile_Async(st.uplo, st.A0.ptr, st.B0.ptr, st.B.ptr, PREC[case["prec"]],
                                                  ctypes.byref(it), ctypes.byref(berr), *s))
        if it.value < 0:
            raise RuntimeError("refinement fell back: ITER %d" % it.value)
    else:
        ch.check(L.CHAMELEON_dlacpy_Tile_Async(ch.UPPERLOWER, st.B0.ptr, st.B.ptr, *s))
        if kind == "posv":
            part = ch.LOWER if st.uplo == ch.LOWER else ch.UPPERLOWER
            ch.check(L.CHAMELEON_dlacpy_Tile_Async(part, st.A0.ptr, st.A.ptr, *s))
            ch.check(L.CHAMELEON_dposv_Tile_Async(st.uplo, st.A.ptr, st.B.ptr, *s))
        else:
            ch.check(L.CHAMELEON_dpotrs_Tile_Async(st.uplo, st.A0.ptr, st.B.ptr, *s))
    ch.check(L.CHAMELEON_Desc_Flush(st.B.ptr, st.seq.ptr))
    ch.check(st.seq.wait())
    return {"x": st.x}


def work(case):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        n, nrhs, source = _systems(case)
        n, nrhs = n.astype(np.float64), nrhs.astype(np.float64)
        own = np.ones(len(n)) if source is None else (source == np.arange(len(n)))
        return {"bytes": float((own * 4.0 * n * (n + 1) + 16.0 * n * nrhs).sum()),
                "flops": float((own * n ** 3 / 3.0 + 2.0 * n * n * nrhs).sum())}
    n, k = float(case["n"]), float(case["nrhs"])
    triangle, rhs = 4.0 * n * (n + 1.0), 16.0 * n * k
    solve = 2.0 * n * n * k
    if kind == "potrs":
        return {"bytes": triangle + rhs, "flops": solve}
    if kind == "mixed":
        return {"bytes": triangle + rhs, "flops": n ** 3 / 3.0 + solve}
    return {"bytes": 2.0 * triangle + rhs, "flops": n ** 3 / 3.0 + solve}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        n, nrhs, source = _systems(case)
        if len(n) > EXACT_MOST_SYSTEMS:
            return None
        xs = []
        for i, (m, k) in enumerate(zip(n.tolist(), nrhs.tolist())):
            src = i if source is None else int(source[i])
            dev = "cuda" if m > 600 else "cpu"
            low = torch.linalg.cholesky(spd_matrix(m, _seed_a(seed) + src, dev))
            x = torch.cholesky_solve(random_matrix(m, k, _seed_b(seed) + i, dev), low)
            xs.append(x.T.contiguous().cpu().numpy().ravel())
        out = {"x": np.concatenate(xs)}
        if kind == "batch":
            out["info"] = None
        return out
    n, k = case["n"], case["nrhs"]
    if kind == "mixed" and n > 8192:
        return None              # the generator of this matrix is the library's own
    if kind == "mixed":
        a = conditioned_matrix(n, case["kappa"], seed)
    else:
        a = spd_matrix(n, _seed_a(seed), "cuda")
    low = torch.linalg.cholesky(a)
    x = torch.cholesky_solve(random_matrix(n, k, _seed_b(seed), "cuda"), low)
    if kind != "lapack":
        return {"x": np.asfortranarray(x.cpu().numpy())}
    up = case["uplo"] == "U"
    a = low.T.triu() + a.tril(-1) if up else low.tril() + a.triu(1)
    return {"a": a.cpu().numpy(), "x": x.cpu().numpy()}
