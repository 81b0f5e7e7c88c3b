/*
 * chol.hip -- FP64 tile kernels of the tiled Cholesky factor-and-solve path
 * for gfx950 (MI355X).  They replace the four tile operations Chameleon
 * submits per step of its right-looking algorithm (compute/pzpotrf.c:84-135:
 * POTRF on A(k,k), TRSM on A(m,k), SYRK on A(n,n), GEMM on A(m,n)) and the
 * tile operations of its triangular solves (compute/pztrsm.c:134-201).
 *
 * All tiles are device mirror tiles: ldt x ldt doubles, column-major,
 * contiguous, ldt a multiple of 16 (see internal.h).
 *
 * Every kernel reads the device info flag first and returns when an earlier
 * diagonal block was found not positive definite, so a failed
 * factorisation stops doing work without a host round trip.
 */
#include "../internal.h"
#include "mfma.h"

namespace chx {
namespace k {

/* ------------------------------------------------------------------ */
/* XCD-aware block order.  Workgroups are dealt to the 8 XCDs of the chip
 * round-robin by id; this remap gives each XCD a contiguous range of logical
 * block ids so that blocks working on the same tiles share an L2.          */
__device__ __forceinline__ int xcd_remap(int id, int total)
{
    const int nx = 8;
    int per = total / nx, rem = total % nx;
    int x = id % nx, local = id / nx;
    return (x < rem) ? x * (per + 1) + local : rem * (per + 1) + (x - rem) * per + local;
}

/* Global -> register load of one K slice (BK rows of W contiguous
 * elements, leading dimension ld) as v2d per thread, and the matching
 * register -> LDS store into a [BK][W] array. */
template <int W, int L, int NTH>
__device__ __forceinline__ void gload_slice(v2d (&r)[L], const double *src, int kb, int ld, int tid)
{
#pragma unroll
    for (int it = 0; it < L; ++it) {
        const int e = (it * NTH + tid) * 2;
        r[it] = *reinterpret_cast<const v2d *>(src + (e % W) + (size_t)(kb + e / W) * ld);
    }
}

template <int W, int L, int NTH>
__device__ __forceinline__ void lstore_slice(double *lds, const v2d (&r)[L], int tid)
{
#pragma unroll
    for (int it = 0; it < L; ++it) {
        const int e = (it * NTH + tid) * 2;
        *reinterpret_cast<v2d *>(lds + e) = r[it];
    }
}

/* ================================================================== */
/* Trailing update of step k: A(m,n) -= A(m,k) A(n,k)^T for the tile pairs
 * (with kp = 2, the two panels k and k+1 at once: A(m,n) -= A(m,k) A(n,k)^T
 * + A(m,k+1) A(n,k+1)^T, one read and write of A(m,n) for both steps)
 * n <= m of either ncol columns n0 .. n0+ncol-1 (ncol > 0, the lookahead
 * columns) or the whole trailing triangle n0 <= n <= m < NT (ncol = 0).
 * Diagonal tiles (m == n) only write their lower triangle: that is the SYRK
 * of pzpotrf.c:112-117, the off-diagonal pairs are its GEMMs
 * (pzpotrf.c:123-129), all in one launch.
 *
 * Block tile BM x BN, K staged through LDS in BK-deep slices with the next PF
 * slices prefetched into registers while one is multiplied.  Each wavefront
 * owns a WM x WN sub-tile of (WM/16)x(WN/16) MFMA blocks; its operand
 * fragments are read from LDS one set (GQ 4-deep steps) ahead of the MFMAs
 * that use them, and the first set of the next slice right after the slice
 * barrier.  Operands are swapped (D = B A^T) so each lane's results are
 * consecutive rows of one column: stores of 16 lanes form one 128-byte
 * segment.
 *
 * The matrix cores bound it.  One wavefront on a SIMD issues an FP64 MFMA
 * every 64 clocks with one LDS read after each product, every 76 with the
 * reads before them and 83 after: the order is asked for where few
 * wavefronts share a SIMD (PF > 1).  The 128 x 128 blocks run four wavefronts
 * on a SIMD, which cover each other, and have no registers for two slices
 * (measured 5 % slower with them).  The order of the sum over k is the same
 * for all block sizes, and so are the results.                            */
template <int BM, int BN, int WM, int WN, int BK, int PF>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64, 2) void trailing_update_kernel(
    double *A, int lmt, int ldt, int k, int kp, int n0, int NT, int ncol, int total_blocks, const int *info,
    const unsigned char *pmap, int atomic_c)
{
    constexpr int NW = (BM / WM) * (BN / WN);
    constexpr int NTH = NW * 64;
    constexpr int FM = WM / 16, FN = WN / 16;
    constexpr int LA = (BK * BM) / (2 * NTH);   /* v2d loads per thread for A */
    constexpr int LB = (BK * BN) / (2 * NTH);
    constexpr int KS = BK / 4;
    static_assert(LA >= 1 && LB >= 1, "tile too small for the thread count");
    static_assert(PF == 1 || PF % 2 == 0, "the unrolled loop keeps the LDS stage static");
    /* two LDS stages: stage s+1 is stored while stage s is multiplied,
     * one barrier per K slice */
    __shared__ double As[2][BK * BM];
    __shared__ double Bs[2][BK * BN];

    const int bad = *info;
    if (PF == 1 && bad != 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int bid = xcd_remap(blockIdx.x, total_blocks);
    const int tbm = ldt / BM, tbn = ldt / BN;
    const int bpt = tbm * tbn;
    const int pair = bid / bpt, b = bid % bpt;
    int m, n;
    if (ncol > 0) {
        /* column n holds the NT - n tiles n .. NT-1 */
        int q = pair, len = NT - n0;
        n = n0;
        while (q >= len && n + 1 < n0 + ncol) {
            q -= len;
            ++n;
            --len;
        }
        m = n + q;
    } else {
        /* pair -> (i, j), i >= j, row-major over the lower triangle */
        int i = (int)((sqrt(8.0 * (double)pair + 1.0) - 1.0) * 0.5);
        while ((long long)(i + 1) * (i + 2) / 2 <= pair) ++i;
        while ((long long)i * (i + 1) / 2 > pair) --i;
        const int j = pair - i * (i + 1) / 2;
        m = n0 + i;
        n = n0 + j;
    }
    /* per-tile precision map: this launch updates the FP64 tiles only */
    if (pmap && pmap[m + (size_t)n * NT] != 0) return;
    const int bi = b % tbm, bj = b / tbm;
    const int row0 = bi * BM, col0 = bj * BN;
    const bool diag = (m == n);
    if (diag && col0 >= row0 + BM) return;

    const size_t ts = (size_t)ldt * ldt;
    const double *Am = A + ((size_t)k * lmt + m) * ts + row0;
    const double *An = A + ((size_t)k * lmt + n) * ts + col0;
    double *C = A + ((size_t)n * lmt + m) * ts;

    const int wm = (wave % (BM / WM)) * WM, wn = (wave / (BM / WM)) * WN;
    v4d acc[FM][FN];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = zero4d();

    v2d ra[PF][LA], rb[PF][LB];
    /* kp panels (1 or 2, tile columns k ..) of ldt / BK slices each */
    const int SK = ldt / BK, S = kp * SK;
    const size_t pstride = (size_t)lmt * ts;
    auto gload = [&](int st, v2d (&xa)[LA], v2d (&xb)[LB]) {
        const int pi = st >= SK, kb = (st - (pi ? SK : 0)) * BK;
        gload_slice<BM, LA, NTH>(xa, Am + pi * pstride, kb, ldt, tid);
        gload_slice<BN, LB, NTH>(xb, An + pi * pstride, kb, ldt, tid);
    };
    auto lstore = [&](int buf, const v2d (&xa)[LA], const v2d (&xb)[LB]) {
        lstore_slice<BM, LA, NTH>(As[buf], xa, tid);
        lstore_slice<BN, LB, NTH>(Bs[buf], xb, tid);
    };
    /* operand fragments of GQ 4-deep steps, two sets */
    constexpr int GQ = (PF > 1 && FM * FN < 4) ? 4 / (FM * FN) : 1, NG = KS / GQ;
    static_assert(KS % GQ == 0 && NG % 2 == 0, "fragment sets alternate within a slice");
    double fa[2][GQ][FM], fb[2][GQ][FN];
    auto fload = [&](int buf, int g, int set) {
        const double *as = As[buf], *bs = Bs[buf];
#pragma unroll
        for (int q = 0; q < GQ; ++q) {
            const int kr = 4 * (g * GQ + q) + (lane >> 4);
#pragma unroll
            for (int fm = 0; fm < FM; ++fm) fa[set][q][fm] = as[kr * BM + wm + fm * 16 + (lane & 15)];
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) fb[set][q][fn] = bs[kr * BN + wn + fn * 16 + (lane & 15)];
        }
    };
    auto multiply = [&](int cur, bool more) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int set = g & 1;
            if (g + 1 < NG) {
                fload(cur, g + 1, set ^ 1);
            } else {
                /* slice st+1 is in LDS and every wave is done reading
                 * slice st (its buffer is refilled next iteration) */
                __syncthreads();
                if (more) fload(cur ^ 1, 0, set ^ 1);
            }
#pragma unroll
            for (int q = 0; q < GQ; ++q)
#pragma unroll
                for (int fm = 0; fm < FM; ++fm)
#pragma unroll
                    for (int fn = 0; fn < FN; ++fn)
                        acc[fm][fn] = mfma_f64(fb[set][q][fn], fa[set][q][fm], acc[fm][fn]);
            if constexpr (PF > 1) {
#pragma unroll
                for (int i = 0; i < GQ * FM * FN; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   /* one product, */
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   /* one LDS read */
                }
            }
        }
    };
    if constexpr (PF == 1) {
        gload(0, ra[0], rb[0]);
        lstore(0, ra[0], rb[0]);
        if (S > 1) gload(1, ra[0], rb[0]);
        __syncthreads();
        fload(0, 0, 0);
        for (int st = 0; st < S; ++st) {
            const int cur = st & 1;
            if (st + 1 < S) {
                lstore(cur ^ 1, ra[0], rb[0]);
                if (st + 2 < S) gload(st + 2, ra[0], rb[0]);
            }
            multiply(cur, st + 1 < S);
        }
    } else {
        /* PF slices in flight: set st % PF holds slice st + 1.  Loads past the
         * end repeat the last slice instead of being skipped, so that no wait
         * for older loads follows a branch. */
        {
            v2d xa[LA], xb[LB];
            gload(0, xa, xb);
#pragma unroll
            for (int j = 0; j < PF; ++j) gload(j + 1 < S ? j + 1 : S - 1, ra[j], rb[j]);
            if (bad != 0) return;
            lstore(0, xa, xb);
        }
        __syncthreads();
        fload(0, 0, 0);
        for (int st = 0; st < S; st += PF) {
#pragma unroll
            for (int j = 0; j < PF; ++j) {
                if (st + j >= S) break;
                lstore((j & 1) ^ 1, ra[j], rb[j]);
                gload(st + j + 1 + PF < S ? st + j + 1 + PF : S - 1, ra[j], rb[j]);
                multiply(j & 1, true);
            }
        }
    }
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int gi = row0 + wm + fm * 16 + (lane & 15);
                const int gj = col0 + wn + fn * 16 + (lane >> 4) + 4 * s;
                if (!diag || gi >= gj) c_sub(&C[gi + (size_t)gj * ldt], acc[fm][fn][s], atomic_c);
            }
}

template <int BM, int BN, int WM, int WN, int BK, int PF>
static void launch_update(double *A, int lmt, int ldt, int k, int kp, int n0, int NT, int ncol, int npairs,
                          const int *info, hipStream_t s, const unsigned char *pmap)
{
    const int bpt = (ldt / BM) * (ldt / BN);
    const long long total = (long long)npairs * bpt;
    if (total <= 0) return;
    constexpr int NTH = (BM / WM) * (BN / WN) * 64;
    hipLaunchKernelGGL((trailing_update_kernel<BM, BN, WM, WN, BK, PF>), dim3((unsigned)total), dim3(NTH), 0, s, A, lmt,
                       ldt, k, kp, n0, NT, ncol, (int)total, info, pmap, atomic_tile_updates());
}

/* the tile updates subtract with FP64 atomic adds in the L2 (c_sub);
 * CHAMAMD_ATOMIC_UPDATE=0: load, subtract and store */
int atomic_tile_updates()
{
    static const int v = [] {
        const char *e = getenv("CHAMAMD_ATOMIC_UPDATE");
        return (e && *e == '0') ? 0 : 1;
    }();
    return v;
}

int update_pairs(int n0, int n1, int NT, int *ncol)
{
    n1 = n1 < NT ? n1 : NT;
    const int S = NT - n0;
    /* columns n0 .. n1-1 only, unless that is the whole triangle */
    const int nc = (n1 < NT || n1 == n0 + 1) ? n1 - n0 : 0;
    *ncol = nc;
    if (nc == 0) return S * (S + 1) / 2;
    return nc * S - nc * (nc - 1) / 2;
}

void trailing_update(double *A, int lmt, int ldt, int k, int n0, int n1, int NT, const int *info, hipStream_t s,
                     int kp, const unsigned char *pmap)
{
    if (n0 >= NT || n1 <= n0) return;
    int ncol = 0;
    const int npairs = update_pairs(n0, n1, NT, &ncol);
    static const int ncu = [] {
        int dev = 0, n = 0;
        CHX_HIP(hipGetDevice(&dev));
        CHX_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
        return n;
    }();
    /* By the launch's work in 64 x 64 blocks: small launches take small
     * blocks, which spread over the compute units and end together, large ones
     * large blocks, which read less.  Whole triangles of S tile columns on 256
     * compute units, times in us with 32 / 64 / 128 blocks:
     *   ldt 256, K 512:  S 8   (576 blocks)   46 /  55 /  80
     *                    S 14  (1680)        128 / 121 / 143
     *                    S 24  (4800)        368 / 313 / 370
     *                    S 50  (20400)      1639 / 1337 / 1336
     *   ldt 512, K 1024: S 8   (2304)        332 / 293 / 394
     *                    S 18  (10944)      1659 / 1378 / 1418
     *                    S 32  (33792)      5314 / 4343 / 4200
     * and one tile column, ldt 320, K 320: 250 blocks 15 / 21 (the 64 x 64
     * blocks as they were before took 22), 50 blocks 7 / 16 (18); ldt 320, S 10,
     * K 640 (1375 blocks) 119 / 128 (133).
     * CHAMAMD_SMALL_COLS=0: launches of single columns take the largest blocks
     * that divide a tile. */
    static const bool small_cols = [] {
        const char *e = getenv("CHAMAMD_SMALL_COLS");
        return !(e && atoi(e) == 0);
    }();
    const bool largest = ncol > 0 && !small_cols;
    const long long b64 = ((long long)npairs * ldt / 64) * ldt / 64;
    if (ldt % 128 == 0 && (largest || b64 >= 80LL * ncu))
        launch_update<128, 128, 32, 64, 16, 1>(A, lmt, ldt, k, kp, n0, NT, ncol, npairs, info, s, pmap);
    else if (ldt % 64 == 0 && (largest || b64 >= 6LL * ncu))
        launch_update<64, 64, 32, 32, 16, 2>(A, lmt, ldt, k, kp, n0, NT, ncol, npairs, info, s, pmap);
    else if (ldt % 32 == 0)
        launch_update<32, 32, 16, 16, 32, 2>(A, lmt, ldt, k, kp, n0, NT, ncol, npairs, info, s, pmap);
    else
        launch_update<16, 16, 16, 16, 16, 1>(A, lmt, ldt, k, kp, n0, NT, ncol, npairs, info, s, pmap);
}

/* ================================================================== */
/* Strided batched GEMM for the solves:
 *   C_j = beta C_j + alpha op(A_j) B_j,   j < batch
 * op(A) is M x K (transA = 0: A(i,p) at A[i + p lda]; 1: at A[p + i lda]),
 * B is K x N with B(p,q) at B[p + q ldb].  M, N, K multiples of the block
 * sizes.  An extra block row (blockIdx.y == batch) copies B_0 into
 * copy_dst (same shape and leading dimension as B) when copy_dst != null,
 * which is how the right-looking solve writes the solved block back while
 * the blocks below are updated with it.                                  */
template <int BM, int BN, int WM, int WN, int TRANSA>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void gemm_batched_kernel(
    int M, int N, int K, double alpha, const double *A0, int lda, long long sA, const double *B0, int ldb,
    long long sB, double beta, double *C0, int ldc, long long sC, int batch, double *copy_dst, const int *info)
{
    constexpr int NW = (BM / WM) * (BN / WN);
    constexpr int NTH = NW * 64;
    constexpr int BK = 16;
    constexpr int FM = WM / 16, FN = WN / 16;
    __shared__ double As[BK][BM + 1];
    __shared__ double Bs[BK][BN + 1];
    if (*info != 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = blockIdx.y;
    const int tbm = M / BM;
    const int bi = blockIdx.x % tbm, bj = blockIdx.x / tbm;
    const int row0 = bi * BM, col0 = bj * BN;
    if (j == batch) {
        /* copy job: B_0 -> copy_dst over this block's region (rows of K) */
        for (int e = tid; e < BM * BN; e += NTH) {
            const int i = row0 + e % BM, q = col0 + e / BM;
            if (i < K && q < N) copy_dst[i + (size_t)q * ldb] = B0[i + (size_t)q * ldb];
        }
        return;
    }
    const double *A = A0 + (size_t)j * sA;
    const double *B = B0 + (size_t)j * sB;
    double *C = C0 + (size_t)j * sC;
    const int wm = (wave % (BM / WM)) * WM, wn = (wave / (BM / WM)) * WN;
    v4d acc[FM][FN];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = zero4d();

    for (int kb = 0; kb < K; kb += BK) {
        /* A slice: op(A)(row0 + i, kb + p) */
        for (int e = tid; e < BK * BM; e += NTH) {
            int i, p;
            double v;
            if (TRANSA) {
                p = e % BK; i = e / BK;
                v = A[(kb + p) + (size_t)(row0 + i) * lda];
            } else {
                i = e % BM; p = e / BM;
                v = A[(row0 + i) + (size_t)(kb + p) * lda];
            }
            As[p][i] = v;
        }
        /* B slice: B(kb + p, col0 + q), K-contiguous */
        for (int e = tid; e < BK * BN; e += NTH) {
            const int p = e % BK, q = e / BK;
            Bs[p][q] = B[(kb + p) + (size_t)(col0 + q) * ldb];
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            double a[FM], bv[FN];
#pragma unroll
            for (int fm = 0; fm < FM; ++fm) a[fm] = As[kk + (lane >> 4)][wm + fm * 16 + (lane & 15)];
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) bv[fn] = Bs[kk + (lane >> 4)][wn + fn * 16 + (lane & 15)];
#pragma unroll
            for (int fm = 0; fm < FM; ++fm)
#pragma unroll
                for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = mfma_f64(bv[fn], a[fm], acc[fm][fn]);
        }
        __syncthreads();
    }
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int gi = row0 + wm + fm * 16 + (lane & 15);
                const int gj = col0 + wn + fn * 16 + (lane >> 4) + 4 * s;
                double *pc = C + gi + (size_t)gj * ldc;
                const double v = alpha * acc[fm][fn][s];
                *pc = (beta == 0.0) ? v : beta * (*pc) + v;
            }
}

template <int BM, int BN, int WM, int WN>
static void launch_gemm(int transA, int M, int N, int K, double alpha, const double *A, int lda, long long sA,
                        const double *B, int ldb, long long sB, double beta, double *C, int ldc, long long sC,
                        int batch, double *copy_dst, const int *info, hipStream_t s)
{
    constexpr int NTH = (BM / WM) * (BN / WN) * 64;
    dim3 grid((M / BM) * (N / BN), batch + (copy_dst ? 1 : 0));
    if (grid.y == 0) return;
    if (transA)
        hipLaunchKernelGGL((gemm_batched_kernel<BM, BN, WM, WN, 1>), grid, dim3(NTH), 0, s, M, N, K, alpha, A, lda,
                           sA, B, ldb, sB, beta, C, ldc, sC, batch, copy_dst, info);
    else
        hipLaunchKernelGGL((gemm_batched_kernel<BM, BN, WM, WN, 0>), grid, dim3(NTH), 0, s, M, N, K, alpha, A, lda,
                           sA, B, ldb, sB, beta, C, ldc, sC, batch, copy_dst, info);
}

void gemm_batched(int transA, int M, int N, int K, double alpha, const double *A, int lda, long long strideA,
                  const double *B, int ldb, long long strideB, double beta, double *C, int ldc, long long strideC,
                  int batch, double *copy_dst, const int *info, hipStream_t s)
{
    if (M % 64 == 0 && N % 64 == 0)
        launch_gemm<64, 64, 32, 32>(transA, M, N, K, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC,
                                    batch, copy_dst, info, s);
    else if (M % 64 == 0 && N % 16 == 0)
        launch_gemm<64, 16, 16, 16>(transA, M, N, K, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC,
                                    batch, copy_dst, info, s);
    else
        launch_gemm<16, 16, 16, 16>(transA, M, N, K, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC,
                                    batch, copy_dst, info, s);
}

} /* namespace k */
} /* namespace chx */
