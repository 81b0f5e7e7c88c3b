/*
 * panel.hip -- the critical-path kernels of the tiled Cholesky on gfx950:
 * POTRF of a diagonal tile (the tile kernel behind INSERT_TASK_dpotrf,
 * coreblas/compute/core_zpotrf.c:75-81, called at compute/pzpotrf.c:90-94)
 * and the panel TRSM (INSERT_TASK_dtrsm(Right, Lower, Trans, NonUnit),
 * pzpotrf.c:99-105), plus the 64 x 64 diagonal-block inverses they share.
 *
 * Both work on 64-column blocks.  POTRF factors a 64-column block of the
 * diagonal tile with a 16-column inner loop (16 x 16 blocks factored in
 * registers by one wavefront) and keeps the inverses of the 16 x 16 blocks,
 * with which the rows below are solved by MFMA products; the explicit inverse
 * of the 64 x 64 block goes to the triangular solves.  The inverses are stored as 64 x 64 column-major blocks, ldt/64
 * (rounded up) per diagonal tile.
 */
#include "../internal.h"
#include "mfma.h"

namespace chx {
namespace k {

#define OB 64       /* outer block width */
#define OBP 65      /* padded LDS row */

/* ------------------------------------------------------------------ */
/* acc[f] += X[0:16, 0:K] * Y[16f:16f+16, 0:K]^T for f < NF, one wavefront;
 * X, Y column-major with leading dimension ld, K a multiple of 16, loads
 * pipelined one 16-deep slice ahead.  Formed as D = Y X^T: lane l holds
 * (row l%16, col 16f + l/16 + 4s) in slot s of acc[f].                    */
template <int NF>
__device__ __forceinline__ void wave_gemm_nt(const double *X, const double *Y, int ld, int K, int lane, v4d *acc)
{
    const int li = lane & 15, lk = lane >> 4;
    if (K <= 0) return;
    const double *px = X + li + (size_t)lk * ld;
    const double *py = Y + li + (size_t)lk * ld;
    double x[4], y[NF][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        x[q] = px[(size_t)(4 * q) * ld];
#pragma unroll
        for (int f = 0; f < NF; ++f) y[f][q] = py[16 * f + (size_t)(4 * q) * ld];
    }
    for (int p = 0; p < K; p += 16) {
        double xn[4], yn[NF][4];
        const bool more = p + 16 < K;
        if (more) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                xn[q] = px[(size_t)(p + 16 + 4 * q) * ld];
#pragma unroll
                for (int f = 0; f < NF; ++f) yn[f][q] = py[16 * f + (size_t)(p + 16 + 4 * q) * ld];
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int f = 0; f < NF; ++f) acc[f] = mfma_f64(y[f][q], x[q], acc[f]);
        if (more) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                x[q] = xn[q];
#pragma unroll
                for (int f = 0; f < NF; ++f) y[f][q] = yn[f][q];
            }
        }
    }
}

__device__ __forceinline__ void wave_gemm_nt_dyn(int nf, const double *X, const double *Y, int ld, int K, int lane,
                                                 v4d *acc)
{
    switch (nf) {
    case 1: wave_gemm_nt<1>(X, Y, ld, K, lane, acc); break;
    case 2: wave_gemm_nt<2>(X, Y, ld, K, lane, acc); break;
    case 3: wave_gemm_nt<3>(X, Y, ld, K, lane, acc); break;
    default: wave_gemm_nt<4>(X, Y, ld, K, lane, acc); break;
    }
}

/* 1/sqrt(d): hardware estimate refined by two Newton-Raphson steps (quadratic
 * convergence from ~2^-22), each r += r/2 (1 - d r^2) with the residual by
 * fused products; the last takes the rounding of d r into it, so that r is
 * within little more than half a unit in the last place (as r (1.5 - d/2 r r) the
 * roundings of the product stayed in it: every solve multiplies by this value
 * twice per row).  NaN and non-positive d propagate as NaN or are caught by the
 * caller's pivot test. */
__device__ __forceinline__ double rsqrt_f64(double d)
{
    double r = __builtin_amdgcn_rsq(d);
    r = fma(0.5 * r, fma(-(d * r), r, 1.0), r);
    const double h = d * r, l = fma(d, r, -h);
    return fma(0.5 * r, fma(-l, r, fma(-h, r, 1.0)), r);
}

/* Column (lane % 16) of the inverse of the lower triangular 16 x 16 block
 * L(r,p) = Ls[r * lds + p], by forward substitution, with the reciprocal
 * diagonal rdiag[r] = 1 / L(r,r). */
__device__ __forceinline__ void block16_inverse_col(const double *Ls, int lds, const double *rdiag, int lane,
                                                    double (&col)[16])
{
    const int jc = lane & 15;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        double s = (r == jc) ? 1.0 : 0.0;
#pragma unroll
        for (int p = 0; p < r; ++p) s -= Ls[r * lds + p] * col[p];
        col[r] = (r < jc) ? 0.0 : s * rdiag[r];
    }
}

/* Inverse Lv of the lower triangular W x W block Ld (W = 16 nfb), given
 * the inverses Lb[I] of its 16 x 16 diagonal blocks, by block rows:
 *   Lv(I,I) = Lb(I),  Lv(I,J) = -Lb(I) sum_{J<=P<I} Ld(I,P) Lv(P,J).
 * Called by the whole workgroup (barriers inside); wavefront J computes
 * block column J. */
__device__ void assemble_inverse(const double (*Ld)[OBP], const double (*Lb)[16][17], double (*Lv)[OBP], int nfb,
                                 int wave, int lane)
{
    const int li = lane & 15, lk = lane >> 4;
    /* diagonal blocks and zero upper blocks */
    for (int e = threadIdx.x; e < OB * OB; e += blockDim.x) {
        const int r = e / OB, c = e % OB;
        const int I = r >> 4, J = c >> 4;
        Lv[r][c] = (I == J && I < nfb) ? Lb[I][r & 15][c & 15] : 0.0;
    }
    __syncthreads();
    for (int I = 1; I < nfb; ++I) {
        const int J = wave;
        if (J < I) {
            v4d S = zero4d();
            for (int P = J; P < I; ++P) {
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
                    S = mfma_f64(Ld[16 * I + li][16 * P + 4 * kk + lk], Lv[16 * P + 4 * kk + lk][16 * J + li], S);
            }
            /* slot kk of S holds S(4kk + lk, li): the B-operand layout */
            v4d R = zero4d();
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) R = mfma_f64(Lb[I][li][4 * kk + lk], S[kk], R);
#pragma unroll
            for (int s = 0; s < 4; ++s) Lv[16 * I + lk + 4 * s][16 * J + li] = -R[s];
        }
        __syncthreads();
    }
}

/* ================================================================== */
/* 64 x 64 diagonal-block inverses of every diagonal tile of a factor that
 * was not produced by potrf_diag in this process.  One workgroup (4
 * wavefronts) per (tile, 64-column block). */
__global__ __launch_bounds__(256) void dinv64_kernel(const double *A, int nt, long long diag_stride, int ldt,
                                                      double *dinv)
{
    __shared__ double Ld[OB][OBP];
    __shared__ double Lv[OB][OBP];
    __shared__ double Lb[4][16][17];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15;
    const int nob = (ldt + OB - 1) / OB;
    const int t = blockIdx.x / nob, C = (blockIdx.x % nob) * OB;
    if (t >= nt) return;
    const int W = min(OB, ldt - C), nfb = W >> 4;
    const double *T = A + (size_t)t * diag_stride;
    for (int e = tid; e < OB * OB; e += 256) {
        const int r = e % OB, c = e / OB;
        Ld[r][c] = (r < W && c < W && r >= c) ? T[(C + r) + (size_t)(C + c) * ldt] : 0.0;
    }
    __syncthreads();
    if (wave < nfb) {
        double col[16], rdiag[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) rdiag[r] = 1.0 / Ld[16 * wave + r][16 * wave + r];
        block16_inverse_col(&Ld[16 * wave][16 * wave], OBP, rdiag, lane, col);
        if (lane < 16) {
#pragma unroll
            for (int q = 0; q < 16; ++q) Lb[wave][q][li] = col[q];
        }
    }
    __syncthreads();
    assemble_inverse(Ld, Lb, Lv, nfb, wave, lane);
    double *dv = dinv + ((size_t)t * nob + C / OB) * OB * OB;
    for (int e = tid; e < OB * OB; e += 256) dv[e] = Lv[e % OB][e / OB];
}

void dinv_all(const double *A, int nt, size_t diag_stride, int ldt, double *dinv, hipStream_t s)
{
    const int nob = (ldt + OB - 1) / OB;
    hipLaunchKernelGGL(dinv64_kernel, dim3(nt * nob), dim3(256), 0, s, A, nt, (long long)diag_stride, ldt, dinv);
}

/* ================================================================== */
/* Right-side triangular solve X = P L^-T, in place, for a batch of tiles.
 * One wavefront owns a 16-row strip of one tile and walks its 64-column
 * blocks left to right:
 *   R = P[:, C:C+64] - X[:, 0:C] L[C:C+64, 0:C]^T    (MFMA, K = C)
 *   X[:, C:C+64] = R Linv_C^T                         (MFMA, K = 64)
 * Tile t uses L0 + t*lstride and the block inverses dinv0 + t*dstride, so
 * applied to identity tiles the kernel forms Linv^T for every diagonal
 * tile at once.                                                          */
__global__ __launch_bounds__(256) void trsm_right_kernel(double *P0, int ntiles, long long pstride, int ldt,
                                                          const double *L0, long long lstride,
                                                          const double *dinv0, long long dstride,
                                                          const int *info)
{
    __shared__ double S[4][16][OBP];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lk = lane >> 4;
    if (*info != 0) return;
    __builtin_amdgcn_s_setprio(2);   /* critical path, see potrf_diag_kernel */
    const int nrb = ldt >> 4;
    const int wid = blockIdx.x * 4 + wave;
    const int t = wid / nrb, rb = wid % nrb;
    if (t >= ntiles) return;
    double *X = P0 + (size_t)t * pstride;
    const double *L = L0 + (size_t)t * lstride;
    const double *dinv = dinv0 + (size_t)t * dstride;
    const int r0 = rb * 16;
    for (int C = 0; C < ldt; C += OB) {
        const int W = min(OB, ldt - C), nfb = W >> 4;
        v4d acc[4] = {zero4d(), zero4d(), zero4d(), zero4d()};
        wave_gemm_nt_dyn(nfb, X + r0, L + C, ldt, C, lane, acc);
        for (int f = 0; f < nfb; ++f)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int c = 16 * f + lk + 4 * s;
                S[wave][li][c] = X[(r0 + li) + (size_t)(C + c) * ldt] - acc[f][s];
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        const double *Lv = dinv + (size_t)(C / OB) * OB * OB;   /* column-major 64 x 64 */
        v4d y[4] = {zero4d(), zero4d(), zero4d(), zero4d()};
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            if (f < nfb) {
#pragma unroll
                for (int kq = 0; kq < 16; ++kq)
                    if (kq < 4 * (f + 1))
                        y[f] = mfma_f64(Lv[(16 * f + li) + (size_t)(4 * kq + lk) * OB], S[wave][li][4 * kq + lk], y[f]);
            }
        }
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            if (f < nfb) {
#pragma unroll
                for (int s = 0; s < 4; ++s) X[(r0 + li) + (size_t)(C + 16 * f + lk + 4 * s) * ldt] = y[f][s];
            }
        }
        __threadfence_block();
        __builtin_amdgcn_wave_barrier();
    }
}

void trsm_right_lower_trans_batched(double *P0, int ntiles, long long pstride, int ldt,
                                    const double *L0, long long lstride, const double *dinv0, long long dstride,
                                    const int *info, hipStream_t s)
{
    if (ntiles <= 0) return;
    const int waves = ntiles * (ldt >> 4);
    const int blocks = (waves + 3) / 4;
    hipLaunchKernelGGL(trsm_right_kernel, dim3(blocks), dim3(256), 0, s, P0, ntiles, pstride, ldt,
                       L0, lstride, dinv0, dstride, info);
}

void trsm_right_lower_trans(double *panel, int ntiles, size_t tile_stride, int ldt, const double *Lkk,
                            const double *dinv, const int *info, hipStream_t s)
{
    trsm_right_lower_trans_batched(panel, ntiles, (long long)tile_stride, ldt, Lkk, 0, dinv, 0, info, s);
}

/* ================================================================== */
/* Fused panel factorisation of step k: POTRF of the diagonal tile
 * (pzpotrf.c:90-94) and the TRSM of the S tiles below it (pzpotrf.c:99-105)
 * in one launch, spread over 64-row units so that the panel is not bounded
 * by one compute unit.
 *
 * What bounds it is the chain of 64 x 64 diagonal factorisations, so one
 * workgroup, the chain, makes all of them and nothing on the way from one
 * to the next goes to another workgroup and back.  Units (one workgroup of 4
 * wavefronts each, ND = ldt / 64 column blocks, in ticket order):
 *   chain       for C = 0 .. ND-1, from D(C) and R(C), which hold A(C, C) and
 *               A(C, C-1) less the products of the column blocks p < C-1:
 *                 X(C, C-1) = R(C) L(C-1, C-1)^-T          (C > 0)
 *                 L(C, C) L(C, C)^T = D(C) - X(C, C-1) X(C, C-1)^T
 *   block (r, C), C < r-1, of the diagonal tile:
 *                 X(r, C) = (A(r, C) - sum_{p<C} X(r, p) X(C, p)^T) L(C, C)^-T
 *               taking each product as its operands are published
 *   R(r), D(r)  the chain's inputs, published while it is on block r-1
 *   the others  one 64-row block below: X(u, C) for every C, left-looking
 * L(C, C) travels as M(C): its 16 x 16 blocks below the diagonal, and the
 * inverses of its four diagonal 16 x 16 blocks.  A product with L(C, C)^-T is
 * then a block substitution on MFMAs whose results stay in registers (the
 * result layout of one product is the operand layout of the next): as many
 * products as with the 64 x 64 inverse, which therefore is off the chain.  It
 * is still wanted (dinv) by the solves: the unit of R(r) forms block r-1's.
 *
 * Measured on MI355X, the launch alone, against one owner per 64 rows with two
 * exchanges per link and the 64 x 64 inverse on the chain (us; tile size, tiles
 * below): 128, 0: 50 -> 36; 256, 27: 109 -> 64; 320, 12: 132 -> 78; 512, 0: 207 ->
 * 103; 512, 30: 227 -> 164; 512, 63: 301 -> 255.  One link is 11.4 us (was 25): 1.2
 * the substitution, 0.9 the first products, 4 x 1.6 the steps (1.2 of it the
 * columns), 3 x 0.5 and 2 x 0.4 the updates and barriers between them.  The other
 * waves' share of each step is cut so that wave 0 never waits for them: it did
 * for 0.8 us in the first and 0.5 in the second step, for the stores behind
 * M(C)'s flag and for R(C+1).  With many tiles below, the FP64 MFMAs are the
 * bound (36 products of 64^3 per row unit, 1.7 us each at the full rate of a
 * compute unit).
 *
 * Publication: a flag set to this launch's epoch after the data was written
 * with device-scope (coherent) stores and every wave has waited for its own
 * to complete (the waves then meet at a barrier, or count themselves in LDS and
 * the last one sets the flag); readers poll the flag
 * and read with device-scope loads, past the non-coherent L2 of other XCDs
 * (a release fence would write back the whole L2 at each link).  Everything
 * published goes through scratch, packed so that 64 units reading one block
 * spread over the memory channels (the tile's 512-byte column pieces, a power
 * of two apart, met on a few of them); the tile's own lines are each
 * touched by one unit of the launch only.
 *
 * Every wait ends.  The units go by level (R(L+1), D(L+1) and the blocks
 * (r, L) for L = 0, 1, ..., then the rows below); the workgroups with tickets
 * 1 .. nw take every nw-th unit of the diagonal tile in that order, and tickets
 * are taken in the order in which workgroups start.  A unit of level L waits
 * for units of lower levels and for the chain's blocks <= L, the chain's block
 * C for units of levels < C: with the chain and the workgroup of the lowest
 * unfinished unit resident one of them can go on, and a workgroup that has not
 * started yet only needs a place that some finished one leaves.  A wait also
 * ends when the info flag is set (a failed pivot) or after a bounded number
 * of polls.                                                                */

#define PF_SPIN_LIMIT (1 << 22)
#define PF_BLK 256                       /* one 16 x 16 block, element (i, j) at i + 16 j   */
#define PF_LOW (10 * PF_BLK)             /* lower blocks of a 64 x 64 block, packed by rows */
#define PF_W (2 * PF_LOW + 4096)         /* scratch of one row block: M | D | R             */
#define PF_X 4096                        /* a published X(r, C), element (i, k) at i + 64 k  */

struct PanelArgs {
    double *T;           /* diagonal tile                                         */
    double *P;           /* first tile below it; tile t at P + t * ts             */
    long long ts;
    int S, ldt, ND;
    int nw;              /* workgroups that share the units of the diagonal tile   */
    double *dinv;        /* Linv_C at dinv + C * 4096, column-major 64 x 64        */
    double *W;           /* published M, D and R of row block r at W + r * PF_W    */
    double *XW;          /* published X(r, C) at XW + (r (r - 1) / 2 + C) * PF_X   */
    int *flags;          /* X(r, C) at r ND + C, M(r) at r ND + r, R(r) at r
                          * (r > 0), D(r) at ND + r (r > 1)                        */
    unsigned *ctr;       /* [0] tickets taken, [1] workgroups finished (both zero
                          * between launches: the last workgroup clears them)      */
    int epoch;
    int *info;
    int iinfo, nvalid;
    PanelLow low;        /* tiles below in a lower precision (panel_factor_kernel<true>)   */
};

/* Buffer accesses relative to a tile: one per-lane offset register, the
 * uniform part of each address in a scalar offset.  aux 16 sets sc1, a
 * device-scope (coherent) access, the form of a relaxed device-scope
 * atomic load or store. */
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t pf_rsrc(const double *p)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), 0, 0x7fffffff, 0x00020000);
}
template <bool DEV = false>
__device__ __forceinline__ double pf_ld(rsrc_t r, int vo, int so)
{
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, DEV ? 16 : 0));
}
__device__ __forceinline__ v2d pf_ld2(rsrc_t r, int vo, int so)
{
    return __builtin_bit_cast(v2d, __builtin_amdgcn_raw_buffer_load_b128(r, vo, so, 0));
}
template <bool DEV = false>
__device__ __forceinline__ void pf_st(double v, rsrc_t r, int vo, int so)
{
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, vo, so, DEV ? 16 : 0);
}

template <bool DEV = false>
__device__ __forceinline__ void pf_st2(v2d v, rsrc_t r, int vo, int so)
{
    typedef unsigned int u4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, vo, so, DEV ? 16 : 0);
}

/* Packed lower blocks.  A block below the diagonal: lane (li, lk) slot s of an
 * MFMA operand, element (li, lk + 4s), is at block + 64 s + lane.  The inverse
 * of a diagonal block has element (r, c) at (r ^ c) + 16 r: lanes on consecutive
 * columns (as pf_col16 leaves it) or on consecutive rows meet different banks. */
__device__ __forceinline__ constexpr int pf_low(int i, int j) { return (i * (i + 1) / 2 + j) * PF_BLK; }
__device__ __forceinline__ int pf_inv(int r, int c) { return (r ^ c) + 16 * r; }

/* One wave's wait for flag idx of this launch; false if the factorisation
 * failed meanwhile (or the poll limit was reached).  The rows below, hundreds
 * of units on one flag, poll more rarely (SLEEP x 64 cycles between polls). */
template <int SLEEP = 1>
__device__ __forceinline__ bool pf_wave_wait(const PanelArgs &a, int idx, int idx2 = -1)
{
    const int at = idx2 >= 0 && (threadIdx.x & 1) ? idx2 : idx;      /* both flags in one load */
    for (int n = 0;; ++n) {
        const bool set = __hip_atomic_load(&a.flags[at], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.epoch;
        if (__ballot(!set) == 0) return true;
        if ((n & 7) == 7 && __hip_atomic_load(a.info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
        if (n > PF_SPIN_LIMIT) {
            atomicCAS(a.info, 0, PANEL_STALLED);
            return false;
        }
        __builtin_amdgcn_s_sleep(SLEEP);
    }
}

/* The same for the workgroup (uniform result), for one or two flags. */
template <int SLEEP = 1>
__device__ __forceinline__ bool pf_wait(const PanelArgs &a, int idx, int tid, int *s_bad, int idx2 = -1)
{
    if (tid < 64) {
        const bool ok = pf_wave_wait<SLEEP>(a, idx, idx2);
        if (tid == 0) *s_bad = !ok;
    }
    __syncthreads();
    const int bad = *s_bad;
    __syncthreads();
    return bad == 0;
}

__device__ __forceinline__ void pf_stores_done() { __builtin_amdgcn_s_waitcnt(0x0F70); }   /* vmcnt(0) */
__device__ __forceinline__ void pf_set(const PanelArgs &a, int idx)
{
    __hip_atomic_store(&a.flags[idx], a.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void pf_publish(const PanelArgs &a, int idx, int tid)
{
    pf_stores_done();
    __syncthreads();
    if (tid == 0) pf_set(a, idx);
}

/* acc[f] += X[16w + i, k] Y[16f + j, k]^T over one 64-column block (wave w,
 * lane (i, j) of the result layout): x[q] = X(16w + li, 4q + lk) in
 * registers, Ys = Y as [k][row] in LDS.  The operands of a step are read
 * while the step before multiplies, and the order is held: left to itself the
 * compiler reads them where they are used, an LDS latency in every two
 * products. */
__device__ __forceinline__ void pf_mma(const double *Ys, int lane, const double (&x)[16], v4d (&acc)[4])
{
    const double *y0 = Ys + (lane >> 4) * 64 + (lane & 15);
    double y[2][4];
#pragma unroll
    for (int f = 0; f < 4; ++f) y[0][f] = y0[16 * f];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        if (q < 15) {
#pragma unroll
            for (int f = 0; f < 4; ++f) y[(q + 1) & 1][f] = y0[256 * (q + 1) + 16 * f];
        }
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[f] = mfma_f64(y[q & 1][f], x[q], acc[f]);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);      /* two LDS reads of two operands each, */
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        if (q < 15) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);  /* four products */
    }
}

/* y <- y L^-T for this wave's 16 rows: slot s of y[f] is column 16f + lk + 4s
 * of row li on entry and return; Ms holds M (packed). */
__device__ __forceinline__ void pf_subst(const double *Ms, int lane, v4d (&y)[4])
{
    const int li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        v4d t = y[f];
        if (f > 0) {
            v4d acc = zero4d();
#pragma unroll
            for (int i = 0; i < f; ++i)
#pragma unroll
                for (int s = 0; s < 4; ++s) acc = mfma_f64(Ms[pf_low(f, i) + 64 * s + lane], y[i][s], acc);
            t = t - acc;
        }
        v4d x = zero4d();
#pragma unroll
        for (int s = 0; s < 4; ++s) x = mfma_f64(Ms[pf_low(f, f) + pf_inv(li, lk + 4 * s)], t[s], x);
        y[f] = x;
    }
}

/* d - (block (i, j) of X X^T), X in LDS as Xs[k][row]: lane (li, lk) slot s
 * is element (li, lk + 4s) of the block.  The products are summed by
 * themselves: taken off one by one, each of the 64 rounded the diagonal, which
 * is large beside them (eight right-hand sides at N = 1500: error of the
 * solution 7.1e-16 so, 5.8e-16 now). */
__device__ __forceinline__ v4d pf_syrk(const double *Xs, int i, int j, int lane, v4d d)
{
    const double *row = Xs + (lane >> 4) * 64 + (lane & 15);
    double xi[2][4], xj[2][4];
    v4d t = zero4d();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        xi[0][q] = row[256 * q + 16 * i];
        xj[0][q] = row[256 * q + 16 * j];
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        if (b < 3) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                xi[(b + 1) & 1][q] = row[256 * (4 * b + 4 + q) + 16 * i];
                xj[(b + 1) & 1][q] = row[256 * (4 * b + 4 + q) + 16 * j];
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) t = mfma_f64(xj[b & 1][q], xi[b & 1][q], t);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) d[s] -= t[s];
    return d;
}

/* Block (i, j) of a 64 x 64 block in Db less what column block c takes off it
 * (summed by itself, as in pf_syrk) */
__device__ __forceinline__ void pf_take16(double *Db, int i, int j, int c, int lane)
{
    v4d x, t = zero4d();
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = Db[pf_low(i, j) + 64 * s + lane];
#pragma unroll
    for (int s = 0; s < 4; ++s) t = mfma_f64(Db[pf_low(j, c) + 64 * s + lane], Db[pf_low(i, c) + 64 * s + lane], t);
#pragma unroll
    for (int s = 0; s < 4; ++s) Db[pf_low(i, j) + 64 * s + lane] = x[s] - t[s];
}

/* Sixteen right-looking columns by one wavefront, rows across the lanes:
 * lanes 0-15 hold the 16 x 16 diagonal block (lower part), the others rows
 * below it or rows of the identity, which turn into P L16^-T and L16^-T.
 * The update of column k by column j is a[k] -= (a[j] / d) a_kj with the
 * pivot d and the unscaled a_kj read from the diagonal lanes: only the
 * reciprocal (estimate, two Newton steps) is between a pivot and the next,
 * and the other lane reads go on beside it; the square roots scale all
 * columns at the end (pf_scale16).  Returns lane j's pivot j, 1 in the others. */
__device__ __forceinline__ double pf_col16(double (&a)[16], int lane)
{
    double dv = 1.0;                     /* lane j: pivot j */
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const double d = readlane_f64(a[j], j);
        double r = __builtin_amdgcn_rcp(d);
        double s[16];
#pragma unroll
        for (int k = j + 1; k < 16; ++k) s[k] = readlane_f64(a[j], k);
        dv = lane == j ? a[j] : dv;
        r = fma(fma(-d, r, 1.0), r, r);
        r = fma(fma(-d, r, 1.0), r, r);
        const double w = -(a[j] * r);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = j + 1; k < 16; ++k) a[k] = fma(w, s[k], a[k]);
    }
    return dv;
}

/* The columns of pf_col16 scaled by the square roots of its pivots; returns the
 * 1-based index of the first non-positive pivot, 0 if none. */
__device__ __forceinline__ int pf_scale16(double (&a)[16], double dv)
{
    const unsigned long long bad = __ballot(!(dv > 0.0));
    const double rs = rsqrt_f64(dv);
#pragma unroll
    for (int j = 0; j < 16; ++j) a[j] *= readlane_f64(rs, j);
    return __builtin_ffsll((long long)bad);
}

/* One 16-column step of a 64 x 64 block whose lower 16 x 16 blocks are in Db,
 * by one wavefront: lane group lk < nr takes block (c + lk, c), group nr rows of
 * the identity (Id, in LDS).  L(c, c) goes to Ld, the blocks below it back to
 * their place, the inverse of L(c, c) to the diagonal one's.  Every lane has one
 * place to read from and one to write to: as three kinds of lanes each with
 * loads, selects and stores of their own, a step was 2.1 us, with 1.2 for the
 * columns; now 1.6.  Returns the failing column or 0.
 * A pivot whose reciprocal leaves the range of the type (it is infinite below
 * 2^-1024) spoils the columns after it.  With one outside [2^-1000, 2^1000), and
 * those that are not positive among them, the step is done again on S A S and
 * the rows below (and of the identity) times S, S the powers of two next to
 * a_qq^-1/2: the factor is S L then, and the rows come out as they should. */
__device__ __forceinline__ int pf_step16(double *Db, double *Ld, const double *Id, int c, int nr, int lane)
{
    const int li = lane & 15, lk = lane >> 4;
    const int low = pf_low(lk < nr ? c + lk : c, c);
    const double *const src = lk < nr ? Db + low : Id;
    double *const dst = (lk == 0 ? Ld + c * PF_BLK : Db + low) + li;
    const int flip = lk == nr ? 15 : 0;      /* the inverse's element (q, li) is at 16 q + (li ^ q) */
    double v[16], dv;
    auto store = [&]() {
        if (lk <= nr) {
#pragma unroll
            for (int q = 0; q < 16; ++q) dst[16 * q + ((li ^ (q & flip)) - li)] = v[q];
        }
    };
    for (bool scaled = false;; scaled = true) {
        int er = 0;                          /* the exponent of this row of S A S */
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = src[li + 16 * q];
        if (scaled) {
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const double d = readlane_f64(v[q], q);
                const int e = d > 0.0 && d < __builtin_inf() ? -(__builtin_amdgcn_frexp_exp(d) >> 1) : 0;
                v[q] = ldexp(v[q], e);
                if (lane == q) er = e;
            }
#pragma unroll
            for (int q = 0; q < 16; ++q) v[q] = ldexp(v[q], er);
        }
        dv = pf_col16(v, lane);
        if (scaled) {
            const int fail = pf_scale16(v, dv);
#pragma unroll
            for (int q = 0; q < 16; ++q) v[q] = ldexp(v[q], -er);
            store();
            return fail;
        }
        /* sign, exponent and the first bits: 2^-1000 is 0x01700000, 2^1000 0x7e700000 */
        const unsigned hi = (unsigned)__double2hiint(dv);
        if (__builtin_expect(__ballot(hi - 0x01700000u >= 0x7e700000u - 0x01700000u) == 0, 1)) break;
    }
    const int fail = pf_scale16(v, dv);
    store();
    return fail;
}

/* The 64 x 64 inverse from M, into dinv (column-major, zeros above the
 * diagonal): Z(J, J) = Lb(J), Z(I, J) = -Lb(I) sum_{J<=P<I} L(I, P) Z(P, J);
 * wave J < 4 forms block column J in registers.  Xs: 32 KB of LDS, on return
 * element (r, c) at (r ^ (c & 15)) + 64 c.  Of dinv, columns and rows from W on
 * are zero. */
template <int NT>
__device__ __forceinline__ void pf_inverse(const double *Ms, double *Xs, double *dinv, int W, int tid, int wave,
                                           int lane)
{
    const int li = lane & 15, lk = lane >> 4;
    v4d z[4];
#pragma unroll
    for (int I = 0; I < 4; ++I) {
        z[I] = zero4d();
        if (I == wave) {
#pragma unroll
            for (int s = 0; s < 4; ++s) z[I][s] = Ms[pf_low(I, I) + pf_inv(lk + 4 * s, li)];
        } else if (I > wave) {
            v4d t = zero4d();
#pragma unroll
            for (int P = 0; P < I; ++P)
#pragma unroll
                for (int s = 0; s < 4; ++s) t = mfma_f64(Ms[pf_low(I, P) + 64 * s + lane], z[P][s], t);
#pragma unroll
            for (int s = 0; s < 4; ++s) z[I] = mfma_f64(-Ms[pf_low(I, I) + pf_inv(li, lk + 4 * s)], t[s], z[I]);
        }
    }
    __syncthreads();
    if (wave < 4) {
#pragma unroll
        for (int I = 0; I < 4; ++I)
#pragma unroll
            for (int s = 0; s < 4; ++s) Xs[((16 * I + lk + 4 * s) ^ li) + 64 * (16 * wave + li)] = z[I][s];
    }
    __syncthreads();
    for (int e = tid; e < 4096; e += NT)
        dinv[e] = (W == 64 || max(e >> 6, e & 63) < W) ? Xs[e ^ ((e >> 6) & 15)] : 0.0;
}

/* M(C) from its scratch into LDS (whole workgroup; barriers by the caller) */
__device__ __forceinline__ void pf_load_m(const double *W, double *Ms, int tid)
{
    const rsrc_t r = pf_rsrc(W);
    double v[10];
#pragma unroll
    for (int b = 0; b < 10; ++b) v[b] = pf_ld<true>(r, tid * 8, b * PF_BLK * 8);
#pragma unroll
    for (int b = 0; b < 10; ++b) Ms[b * PF_BLK + tid] = v[b];
}

__device__ __forceinline__ double *pf_xw(const PanelArgs &a, int r, int C)
{
    return a.XW + ((size_t)(r * (r - 1) / 2) + C) * PF_X;
}

struct PanelLds {
    double Xs[4096];
    double B[2][PF_LOW];
    double Id[PF_BLK];       /* identity */
    int s_int, s_fail, s_parts;
};

/* the chain (see above) */
__device__ __forceinline__ void panel_chain(const PanelArgs &a, PanelLds &L)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const int ldt = a.ldt, ND = a.ND;
    double *const Xs = L.Xs;
    if (tid == 0) L.s_fail = L.s_int = L.s_parts = 0;
    L.Id[tid] = (tid & 15) == (tid >> 4) ? 1.0 : 0.0;
    /* R(C) and D(C): rv this wave's rows of R, dcol block (wave, 0) of D, drest
     * blocks (wave, 1) and the wave-th of (2,2), (3,2), (3,3); block rows 0 and
     * 1 come from the tile, the others from their units */
    v4d rv[4], dcol = zero4d(), drest[2] = {zero4d(), zero4d()};
    const int r2i = wave == 1 ? 2 : 3, r2j = wave == 3 ? 3 : 2;
    const int vt = (li + lk * ldt) * 8;
    auto tile_at = [&](int i, int j) { return (16 * i + 16 * j * ldt) * 8; };
    int cur = 0;
    for (int C = 0; C < ND; ++C, cur ^= 1) {
        /* Ms: M(C-1), then R(C+1)'s and D(C+1)'s values for wave 0, and from Ld
         * on the diagonal 16 x 16 blocks of L(C, C) */
        double *const Db = L.B[cur], *const Ms = L.B[cur ^ 1], *const Ld = Ms + PF_LOW - 4 * PF_BLK;
        const rsrc_t rM = pf_rsrc(a.W + (size_t)C * PF_W);
        const rsrc_t rD = pf_rsrc(a.T + 64 * C + (size_t)64 * C * ldt);     /* the diagonal block in the tile */
        /* a finished block of M to its scratch, and of L to the tile */
        auto publish = [&](int i, int j) {
            v2d m[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) m[h] = *reinterpret_cast<const v2d *>(Db + pf_low(i, j) + 128 * h + 2 * lane);
#pragma unroll
            for (int h = 0; h < 2; ++h) pf_st2<true>(m[h], rM, lane * 16, (pf_low(i, j) + 128 * h) * 8);
            if (i > j) {
                const int v2 = (2 * (lane & 7) + (lane >> 3) * ldt) * 8;
#pragma unroll
                for (int h = 0; h < 2; ++h) pf_st2(m[h], rD, v2, tile_at(i, j) + 64 * h * ldt);
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const double y = Ld[j * PF_BLK + 64 * s + lane];
                    if (li >= lk + 4 * s) pf_st(y, rD, vt, tile_at(j, j) + 32 * s * ldt);
                }
            }
        };
        if (C == 0) {
            double d[10];
            const int vo = ((tid & 15) + (tid >> 4) * ldt) * 8;
#pragma unroll
            for (int b = 0; b < 10; ++b) {
                const int i = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3, j = b - i * (i + 1) / 2;
                d[b] = pf_ld(rD, vo, tile_at(i, j));
            }
#pragma unroll
            for (int b = 0; b < 10; ++b) Db[b * PF_BLK + tid] = d[b];
            __syncthreads();
        } else {
            if (wave == 0) {
                /* fetched by the other waves while this one was factoring */
#pragma unroll
                for (int q = 0; q < 16; ++q) rv[q >> 2][q & 3] = Db[q * 64 + lane];
#pragma unroll
                for (int s = 0; s < 4; ++s) dcol[s] = Db[(16 + s) * 64 + lane];
            }
            pf_subst(Ms, lane, rv);
            if (wave == 1) {
                pf_stores_done();
                if (lane == 0) pf_set(a, (C - 1) * (ND + 1));
            }
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int s = 0; s < 4; ++s) Xs[(16 * f + lk + 4 * s) * 64 + 16 * wave + li] = rv[f][s];
            __syncthreads();
            {
                const v4d x = pf_syrk(Xs, wave, 0, lane, dcol);
#pragma unroll
                for (int s = 0; s < 4; ++s) Db[pf_low(wave, 0) + 64 * s + lane] = x[s];
            }
            __syncthreads();
        }
        /* factor the 64 x 64 block in Db, by 16-column steps: wave 0 the
         * columns, the others what comes after them and the traffic */
#pragma unroll 1
        for (int cb = 0; cb < 4; ++cb) {
            /* wave 3 repeats the first block during the second step, for its
             * inverse: in the first there is no lane left for the identity */
            if (wave == 0 || (wave == 3 && cb == 1)) {
                const int c = wave == 0 ? cb : 0;
                const int fail = pf_step16(Db, Ld, L.Id, c, wave == 0 ? 4 - cb : 1, lane);
                /* (the padding's own pivots do not count) */
                const int col = 64 * C + 16 * c + fail;
                if (lane == 0 && fail && col - 1 < a.nvalid) L.s_fail = col;
            } else if (cb == 0) {
                if (C > 0) {
                    /* publish X(C, C-1) (R(C+1) waits for it), element (row lane, column k) */
                    const rsrc_t rP = pf_rsrc(pf_xw(a, C, C - 1));
                    v2d xp[11];
#pragma unroll
                    for (int u = 0; u < 11; ++u) xp[u] = *reinterpret_cast<const v2d *>(Xs + 128 * min(3 * u + wave - 1, 31) + 2 * lane);
#pragma unroll
                    for (int u = 0; u < 11; ++u) pf_st2<true>(xp[u], rP, lane * 16, min(3 * u + wave - 1, 31) * 1024);
                    /* the products of column 1, and of (3, 3); in between, the
                     * last wave whose part of X is out sets its flag */
                    const v4d x = pf_syrk(Xs, wave, 1, lane, drest[0]);
#pragma unroll
                    for (int s = 0; s < 4; ++s) Db[pf_low(wave, 1) + 64 * s + lane] = x[s];
                    pf_stores_done();
                    if (lane == 0 && __hip_atomic_fetch_add(&L.s_parts, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 3 * C - 1)
                        pf_set(a, C * ND + C - 1);
                    if (wave == 3) {
                        const v4d y = pf_syrk(Xs, 3, 3, lane, drest[1]);
#pragma unroll
                        for (int s = 0; s < 4; ++s) Db[pf_low(3, 3) + 64 * s + lane] = y[s];
                    }
                }
            } else {
                if (cb == 1 && C > 0) {
                    /* X(C, C-1) to the tile, two columns a store */
                    const rsrc_t rX = pf_rsrc(a.T + 64 * C + (size_t)64 * (C - 1) * ldt);
                    const int vx = (lane & 31) * 16 + (lane >> 5) * ldt * 8;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        v2d xp[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u)
                            xp[u] = *reinterpret_cast<const v2d *>(Xs + 128 * (16 * (wave - 1) + 8 * h + u) + 2 * lane);
#pragma unroll
                        for (int u = 0; u < 8; ++u)
                            pf_st2(xp[u], rX, vx, (16 * (wave - 1) + 8 * h + u) * 16 * ldt);
                    }
                    /* the products of (2, 2) and (3, 2) */
                    const v4d x = pf_syrk(Xs, r2i, 2, lane, drest[1]);
#pragma unroll
                    for (int s = 0; s < 4; ++s) Db[pf_low(r2i, 2) + 64 * s + lane] = x[s];
                }
                if (cb < 3) {
                    /* what step cb-1 takes off the columns after cb: (2,2),
                     * (3,2), (3,3), then (3,3) */
                    for (int u = wave - 1; u < (cb == 1 ? 3 : 1); u += 2) {
                        const int i = u == 0 && cb == 1 ? 2 : 3, j = u == 2 || cb == 2 ? 3 : 2;
                        pf_take16(Db, i, j, cb - 1, lane);
                    }
                }
                /* publish the finished columns of M and store them to the
                 * tile: 0 and 1 beside step 2 (waves 2 and 3), 2 beside step 3 */
                const int j = cb == 2 ? wave - 2 : cb == 3 && wave == 3 ? 2 : -1;
                if (j >= 0)
                    for (int i = j; i < 4; ++i) publish(i, j);
                if (cb == 3 && C + 1 < ND) {
                    /* R(C+1) and D(C+1), wave 0's share among them */
                    bool ok = true;
                    rsrc_t rr, rd;
                    int vo, sr, sd;      /* strides of one slot */
                    if (C == 0) {                /* no products yet: from the tile */
                        rr = pf_rsrc(a.T + 64);
                        rd = pf_rsrc(a.T + 64 + (size_t)64 * ldt);
                        vo = vt; sr = sd = 32 * ldt;
                    } else {
                        ok = pf_wave_wait(a, C + 1, ND + C + 1);
                        rr = pf_rsrc(a.W + (size_t)(C + 1) * PF_W + 2 * PF_LOW);
                        rd = pf_rsrc(a.W + (size_t)(C + 1) * PF_W + PF_LOW);
                        vo = lane * 8; sr = sd = 512;
                    }
                    auto at_r = [&](int w) { return C == 0 ? 128 * w : w * 16 * 512; };
                    auto at_d = [&](int i, int j) { return C == 0 ? tile_at(i, j) : pf_low(i, j) * 8; };
                    if (ok) {
#pragma unroll
                        for (int q = 0; q < 16; ++q) rv[q >> 2][q & 3] = pf_ld<true>(rr, vo, at_r(wave) + q * sr);
#pragma unroll
                        for (int s = 0; s < 4; ++s) {
                            dcol[s] = pf_ld<true>(rd, vo, at_d(wave, 0) + s * sd);
                            drest[0][s] = pf_ld<true>(rd, vo, at_d(wave, 1) + s * sd);
                            drest[1][s] = pf_ld<true>(rd, vo, at_d(r2i, r2j) + s * sd);
                        }
                        double t[7];
#pragma unroll
                        for (int u = 0; u < 7; ++u) {
                            const int q = (wave - 1) * 7 + u;
                            t[u] = q < 16 ? pf_ld<true>(rr, vo, at_r(0) + q * sr)
                                          : pf_ld<true>(rd, vo, at_d(0, 0) + (q < 20 ? q - 16 : 0) * sd);
                        }
#pragma unroll
                        for (int u = 0; u < 7; ++u) Ms[((wave - 1) * 7 + u) * 64 + lane] = t[u];
                    } else if (lane == 0) {
                        L.s_int = 1;
                    }
                }
            }
            if (cb == 3) pf_stores_done();                  /* M's columns */
            __syncthreads();
            if (L.s_fail) break;
            if (cb < 3) {
                /* column cb+1 takes off step cb: block (cb + 1 + wave, cb + 1) */
                const int i = cb + 1 + wave;
                if (i < 4) {
                    pf_take16(Db, i, cb + 1, cb, lane);
                }
                __syncthreads();
            }
        }
        if (L.s_fail) {
            if (tid == 0) atomicCAS(a.info, 0, a.iinfo + L.s_fail);
            return;
        }
        if (L.s_int) return;
        /* the flag of M(C) follows when the stores are done, in the next link */
        if (wave == 1) publish(3, 3);
    }
    if (wave == 1) {
        pf_stores_done();
        if (lane == 0) pf_set(a, (ND - 1) * (ND + 1));
    }
    pf_inverse<256>(L.B[cur ^ 1], Xs, a.dinv + (size_t)(ND - 1) * 4096, 64, tid, wave, lane);
}

/* Block (r, C) of the diagonal tile below its diagonal blocks; for C = r-1 it
 * is R(r), left to the chain's substitution, and the 64 x 64 inverse of block
 * r-1 is formed after it. */
__device__ __forceinline__ void panel_block(const PanelArgs &a, PanelLds &L, int r, int C)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const int ldt = a.ldt, ND = a.ND;
    const bool is_r = C == r - 1;
    const rsrc_t rx = pf_rsrc(a.T + 64 * r + (size_t)64 * C * ldt);
    const int vx = (16 * wave + li + lk * ldt) * 8, c4 = 4 * ldt * 8;
    const int vp = (16 * wave + li + 64 * lk) * 8;      /* (16w + li, lk) of a published block */
    v4d y[4];
    if (r > 1) {
        double av[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) av[q] = pf_ld(rx, vx, q * c4);
        v4d acc[4] = {zero4d(), zero4d(), zero4d(), zero4d()};
        for (int p = 0; p < C; ++p) {
            if (!pf_wait(a, r * ND + p, tid, &L.s_int, C * ND + p)) return;
            double x[16], yst[16];
#pragma unroll
            for (int h = 0; h < 16; ++h) yst[h] = pf_ld<true>(pf_rsrc(pf_xw(a, C, p)), tid * 8, h * 2048);
#pragma unroll
            for (int q = 0; q < 16; ++q) x[q] = pf_ld<true>(pf_rsrc(pf_xw(a, r, p)), vp, q * 2048);
#pragma unroll
            for (int h = 0; h < 16; ++h) L.Xs[tid + 256 * h] = yst[h];
            __syncthreads();
            pf_mma(L.Xs, lane, x, acc);
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) y[q >> 2][q & 3] = av[q] - acc[q >> 2][q & 3];
    }
    if (is_r) {
        if (r > 1) {
            const rsrc_t rW = pf_rsrc(a.W + (size_t)r * PF_W + 2 * PF_LOW);
#pragma unroll
            for (int q = 0; q < 16; ++q) pf_st<true>(y[q >> 2][q & 3], rW, lane * 8, (16 * wave + q) * 512);
            pf_publish(a, r, tid);
        }
    }
    if (!pf_wait(a, C * (ND + 1), tid, &L.s_int)) return;
    pf_load_m(a.W + (size_t)C * PF_W, L.B[0], tid);
    __syncthreads();
    if (is_r) {
        pf_inverse<256>(L.B[0], L.Xs, a.dinv + (size_t)C * 4096, 64, tid, wave, lane);
        return;
    }
    pf_subst(L.B[0], lane, y);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        pf_st<true>(y[q >> 2][q & 3], pf_rsrc(pf_xw(a, r, C)), vp, q * 2048);
        pf_st(y[q >> 2][q & 3], rx, vx, q * c4);
    }
    pf_publish(a, r * ND + C, tid);
}

/* D(r) = A(r, r) - sum_{p < r-1} X(r, p) X(r, p)^T, lower blocks */
__device__ __forceinline__ void panel_diag(const PanelArgs &a, PanelLds &L, int r)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const int ldt = a.ldt, ND = a.ND;
    const rsrc_t rx = pf_rsrc(a.T + 64 * r + (size_t)64 * r * ldt);
    v4d d[3];
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        const int b = min(4 * u + wave, 9), i = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3, j = b - i * (i + 1) / 2;
#pragma unroll
        for (int s = 0; s < 4; ++s) d[u][s] = pf_ld(rx, (16 * i + li + lk * ldt) * 8, (16 * j + 4 * s) * ldt * 8);
    }
    for (int p = 0; p < r - 1; ++p) {
        if (!pf_wait(a, r * ND + p, tid, &L.s_int)) return;
        double yst[16];
#pragma unroll
        for (int h = 0; h < 16; ++h) yst[h] = pf_ld<true>(pf_rsrc(pf_xw(a, r, p)), tid * 8, h * 2048);
#pragma unroll
        for (int h = 0; h < 16; ++h) L.Xs[tid + 256 * h] = yst[h];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            const int b = min(4 * u + wave, 9), i = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3, j = b - i * (i + 1) / 2;
            d[u] = pf_syrk(L.Xs, i, j, lane, d[u]);
        }
    }
    const rsrc_t rW = pf_rsrc(a.W + (size_t)r * PF_W + PF_LOW);
#pragma unroll
    for (int u = 0; u < 3; ++u)
        if (4 * u + wave < 10) {
#pragma unroll
            for (int s = 0; s < 4; ++s) pf_st<true>(d[u][s], rW, lane * 8, ((4 * u + wave) * PF_BLK + 64 * s) * 8);
        }
    pf_publish(a, ND + r, tid);
}

/* The finished columns of block C of a 64-row unit u below (panel_rows' y) in
 * the precision of the trailing products, from registers: a launch that read
 * them back took 5 us of the chain at 256-row tiles and up to 68, beside a bulk
 * update, at 512.  FP32 in the layout of the tile; BF16 row-major, a
 * wavefront's 16 rows turned in its own part of Xs, which is idle between the
 * last product and the next staging. */
__device__ __forceinline__ void panel_low(const PanelArgs &a, PanelLds &L, const v4d (&y)[4], int u, int C, int wave,
                                          int lane)
{
    const int li = lane & 15, lk = lane >> 4, ldt = a.ldt;
    const size_t tile = (size_t)(u / a.ND) * a.ts;
    const int row = 64 * (u % a.ND) + 16 * wave;
    if (a.low.f32) {
        const rsrc_t r = pf_rsrc(reinterpret_cast<const double *>(a.low.f32 + tile + (size_t)64 * C * ldt));
        const int vo = (row + li + lk * ldt) * 4;
#pragma unroll
        for (int q = 0; q < 16; ++q)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint((float)y[q >> 2][q & 3]), r, vo, q * 16 * ldt, 0);
    }
    if (a.low.hi) {
        /* rows of 72 halfwords, so that 16-byte pieces stay aligned */
        unsigned short *const S = reinterpret_cast<unsigned short *>(L.Xs + 1024 * wave);
        for (int plane = 0; plane < (a.low.lo ? 2 : 1); ++plane) {
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const double v = y[q >> 2][q & 3];
                unsigned short b = bf16_bits((float)v);
                if (plane) b = bf16_bits((float)(v - (double)bf16_to_float(b)));
                S[72 * li + 4 * q + lk] = b;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            const rsrc_t r = pf_rsrc(reinterpret_cast<const double *>((plane ? a.low.lo : a.low.hi) + tile + (size_t)row * ldt));
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int i = (lane >> 3) + 8 * h, c = 8 * (lane & 7);
                v2d w;
                __builtin_memcpy(&w, S + 72 * i + c, sizeof w);
                pf_st2(w, r, (i * ldt + c) * 2, 64 * C * 2);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
}

/* X(u, C) of the 64 rows of unit u in the tiles below, every C, left-looking.  The
 * published blocks X(C, p) go through two LDS buffers, one barrier per block;
 * the loads of a block (and of the unit's own X(u, p)) are issued before the
 * products of the one before.  A product is 1.7 us of MFMAs. */
template <bool LOW>
__device__ __forceinline__ void panel_rows(const PanelArgs &a, PanelLds &L, int u)
{
    double *const Rw = a.P + (size_t)(u / a.ND) * a.ts + 64 * (u % a.ND);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const int ldt = a.ldt, ND = a.ND;
    /* offsets from column block p of the rows: those from the first one would
     * pass 32 bits in tiles beyond 16384 */
    auto block = [&](int p) { return pf_rsrc(Rw + (size_t)64 * p * ldt); };
    const int vr = (16 * wave + li + lk * ldt) * 8, c4 = 4 * ldt * 8;
    for (int C = 0; C < ND; ++C) {
        const rsrc_t rC = block(C);
        v4d acc[4] = {zero4d(), zero4d(), zero4d(), zero4d()}, y[4];
        double av[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) av[q] = pf_ld(rC, vr, q * c4);
        if (C > 0) {
            const rsrc_t ry = pf_rsrc(pf_xw(a, C, 0));
            double x[16], yst[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) x[q] = pf_ld(block(0), vr, q * c4);
            /* X(C, C-2) is published after every X(C, p) before it; X(C, C-1)
             * comes last, from the chain */
            if (!pf_wait<16>(a, C * ND + max(C - 2, 0), tid, &L.s_int)) return;
#pragma unroll
            for (int h = 0; h < 16; ++h) yst[h] = pf_ld<true>(ry, tid * 8, h * 2048);
#pragma unroll
            for (int h = 0; h < 16; ++h) L.Xs[tid + 256 * h] = yst[h];
            __syncthreads();
            for (int p = 0; p < C; ++p) {
                double *const cur = p & 1 ? L.B[0] : L.Xs, *const nxt = p & 1 ? L.Xs : L.B[0];
                double xn[16];
                if (p + 1 < C) {
                    if (p + 2 == C && !pf_wait<16>(a, C * ND + C - 1, tid, &L.s_int)) return;
#pragma unroll
                    for (int h = 0; h < 16; ++h) yst[h] = pf_ld<true>(ry, tid * 8, (p + 1) * PF_X * 8 + h * 2048);
#pragma unroll
                    for (int q = 0; q < 16; ++q) xn[q] = pf_ld(block(p + 1), vr, q * c4);
                }
                pf_mma(cur, lane, x, acc);
                if (p + 1 < C) {
#pragma unroll
                    for (int h = 0; h < 16; ++h) nxt[tid + 256 * h] = yst[h];
#pragma unroll
                    for (int q = 0; q < 16; ++q) x[q] = xn[q];
                }
                __syncthreads();
            }
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) y[q >> 2][q & 3] = av[q] - acc[q >> 2][q & 3];
        if (!pf_wait<16>(a, C * (ND + 1), tid, &L.s_int)) return;
        pf_load_m(a.W + (size_t)C * PF_W, L.B[0], tid);
        __syncthreads();
        pf_subst(L.B[0], lane, y);
#pragma unroll
        for (int q = 0; q < 16; ++q) pf_st(y[q >> 2][q & 3], rC, vr, q * c4);
        if constexpr (LOW) panel_low(a, L, y, u, C, wave, lane);
    }
}

/* units of the diagonal tile besides the chain: level L < ND-1 holds R(L+1),
 * D(L+1) (L > 0) and the blocks (r, L), r > L+1 */
__host__ __device__ __forceinline__ int panel_units(int ND) { return ND > 1 ? ND * (ND - 1) / 2 + ND - 2 : 0; }

template <bool LOW>
__global__ __launch_bounds__(256, 2) void panel_factor_kernel(PanelArgs a)
{
    __shared__ PanelLds L;
    __shared__ int s_ticket, s_info;
    const int tid = threadIdx.x;
    __builtin_amdgcn_s_setprio(2);        /* critical path: win issue next to update waves */
    if (tid == 0) {
        s_ticket = (int)atomicAdd(&a.ctr[0], 1u);
        s_info = __hip_atomic_load(a.info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(s_ticket), nu = panel_units(a.ND);
    /* a ticket past the grid would mean the counters were not cleared */
    if (t >= (int)gridDim.x) {
        if (tid == 0) atomicCAS(a.info, 0, PANEL_STALLED);
    } else if (s_info == 0) {
        if (t == 0) {
            panel_chain(a, L);
        } else if (t <= a.nw) {
            for (int i = t - 1; i < nu; i += a.nw) {
                int u = i, lev = 0;
                for (int len = a.ND - 1; u >= len; len = a.ND - lev) {
                    u -= len;
                    ++lev;
                }
                __syncthreads();         /* the last unit is done with the LDS */
                if (lev > 0 && u == 1) panel_diag(a, L, lev + 1);
                else panel_block(a, L, lev + 1 + (u > 1 ? u - (lev > 0) : u), lev);
            }
        } else {
            panel_rows<LOW>(a, L, t - 1 - a.nw);
        }
    }
    __syncthreads();
    if (tid == 0 && atomicAdd(&a.ctr[1], 1u) == gridDim.x - 1) {
        __hip_atomic_store(&a.ctr[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&a.ctr[1], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

size_t panel_scratch(int ldt)
{
    const size_t n = ldt / 64;
    return n * PF_W + n * (n - 1) / 2 * PF_X;
}
int panel_flags(int ldt) { return (ldt / 64) * (ldt / 64) + 1; }

void panel_factor(double *T, double *P, long long ts, int S, int ldt, double *dinv, double *scratch, int *flags,
                  unsigned *ctr, int epoch, int *info, int iinfo, int nvalid, hipStream_t s, const PanelLow &low)
{
    PanelArgs a;
    a.low = low;
    a.T = T; a.P = P; a.ts = ts; a.S = S; a.ldt = ldt; a.ND = ldt / 64;
    a.dinv = dinv; a.W = scratch; a.XW = scratch + (size_t)a.ND * PF_W; a.flags = flags; a.ctr = ctr; a.epoch = epoch;
    a.info = info; a.iinfo = iinfo; a.nvalid = nvalid;
    /* As many workgroups as there are units of the diagonal tile, but no more
     * than leave every 64-row unit below a compute unit of its own, or where
     * those are too many a place of its own (two on a compute unit), as long
     * as there are seven: two row units on one compute unit take twice as
     * long, and one that starts when another has ended doubles the launch
     * (512-column tile, 30 tiles below: 225 us with 33 workgroups, 166 with
     * 15; 63 tiles below: 340 us with 33, 256 with 7). */
    static const int ncu = [] {
        int dev = 0, n = 0;
        CHX_HIP(hipGetDevice(&dev));
        CHX_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
        return n;
    }();
    const int nu = panel_units(a.ND), least = nu < 7 ? nu : 7, rows = 1 + a.ND * S;
    const int room = rows + least <= ncu ? ncu - rows : rows + least <= 2 * ncu ? 2 * ncu - rows : nu;
    a.nw = nu < room ? nu : room;
    const int grid = 1 + a.nw + a.ND * S;
    hipLaunchKernelGGL((low.f32 || low.hi ? panel_factor_kernel<true> : panel_factor_kernel<false>), dim3(grid), dim3(256), 0, s, a);
}

/* ================================================================== */
/* POTRF of one matrix held in HBM per job, one workgroup of 4 or 8 wavefronts
 * per job: the diagonal tile of the tiled factorisation (one job), or
 * every system of a batch (jobs taken from a queue).
 * For each 64-column block C (left-looking):
 *   (a) diagonal block -= T[C:C+64, 0:C] T[C:C+64, 0:C]^T, into LDS (MFMA)
 *   (b) factor the 64 x 64 diagonal block in LDS by 16-column steps, the
 *       inverses of its 16 x 16 diagonal blocks beside them
 *   (c) build the 64 x 64 inverse, store it in dinv
 *   (d) rows below: the products of (a) and X = P L^-T in one pass (MFMA)
 * The strictly upper triangle of the matrix is never written.  A failed
 * job reports the 1-based column of its first non-positive pivot, only
 * for pivots inside its valid part (nvalid columns).
 *
 * A large batch is bound by (d): its operands come from beyond the L2 (512
 * systems are in work at once), so what counts is how far ahead they are asked
 * for and how often they are read.  A wavefront takes two 16-row blocks against
 * the same 64 shared rows, keeps four slices of both in flight, and solves its
 * rows while they are in registers; the rows' old values come as the slices
 * after the last, behind the products.  With one block, one slice, a pass of
 * its own for the solves and the old values asked for at the end, the 20 000
 * systems of orders 16 to 1023 took 24.0 ms, now 16.6; 1024 of order 1024 11.4
 * and 8.5 ms (about 4 TB/s), 2048 of order 512 4.1 and 2.76, 4000 of order 300
 * 1.76 and 1.70 by the old values alone.
 * A small batch is bound by the serial (b), 18 us per block before and 9 now
 * (the steps of the panel's chain): 4000 of order 64 366 and 178 us, one of
 * order 256 198 and 115. */

struct PotrfJobs {
    double *A;               /* job j: matrix at A + off[j] (off null: A)               */
    const long long *off;
    const int *np;           /* order (multiple of 16); null: np0                        */
    const int *ld;           /* leading dimension; null: ld0, or np when ld0 = 0         */
    const int *nvalid;       /* valid columns; null: nvalid0                             */
    double *dinv;            /* 64 x 64 inverses: job j at dinv + doff[j] (null: dinv)   */
    const long long *doff;
    int np0, ld0, nvalid0;
    int count;               /* number of jobs                                           */
    int *queue;              /* job counter (batches); null: job = blockIdx.x            */
    int *info;               /* single job: *info = iinfo + column on failure;
                              * batches: info[j] = column or 0                           */
    int iinfo, batch;
};

/* Products of the 16-row blocks rb0 + wave + NW u, u < NB, of the nrb from row
 * C on, and what follows them: DIAG, the diagonal block's (NB = 1, four
 * wavefronts), goes to Db; rows below are solved with M in Db and stored.  The
 * 16-deep slices of the 64 shared rows (Y) are staged in LDS, double-buffered;
 * every wavefront streams its own rows (X; DIAG reads them from Y).  C is a
 * multiple of 64, so the ring of four slices needs no test, and the four slices
 * after the last hold the old values of the block's own columns: they are in
 * flight behind the last products (DIAG loads those of its lower blocks at the
 * start).  Shared rows past the last slice repeat it.  A block past the matrix reads rows li instead, and
 * shared rows past the matrix (last block column) whatever follows in it:
 * neither is used.  FP32 products leave other columns in a slot than FP64
 * ones; their shared rows are read in an order (pi) that undoes it. */
template <int NW, int NB, bool LP, bool DIAG>
__device__ __forceinline__ void jobs_update(double *T, int ldt, int C, int rb0, int nrb, double *Ys, double *Db,
                                            int tid)
{
    constexpr int NT = NW * 64, YH = 512 / NT;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lk = lane >> 4;
    const int pi = LP ? (li >> 2) + 4 * (li & 3) : li;
    const int S = C >> 4;
    /* offsets from the first column of a slice, whose address is a scalar */
    int vx[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        const int rb = rb0 + wave + NW * u;
        vx[u] = ((rb < nrb ? C + 16 * rb + li : li) + lk * ldt) * 8;
    }
    const int vy = (C + (tid & 31) * 2 + (tid >> 5) * ldt) * 8;
    double *const ys = Ys + (tid >> 5) * OB + (tid & 31) * 2;
    v4d acc[NB][4];
    v4f accf[NB][4];
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            acc[u][f] = zero4d();
            accf[u][f] = zero4f();
        }
    v2d y[4][YH];
    double x[4][NB][4];
    auto yload = [&](int st, v2d (&r)[YH]) {
        const rsrc_t b = pf_rsrc(T + (size_t)(16 * min(st, S - 1)) * ldt);
#pragma unroll
        for (int h = 0; h < YH; ++h) r[h] = pf_ld2(b, vy, h * (NT / 4) * ldt);
    };
    auto ystore = [&](int buf, const v2d (&r)[YH]) {
#pragma unroll
        for (int h = 0; h < YH; ++h) *reinterpret_cast<v2d *>(ys + buf * 16 * OB + h * (NT / 32) * OB) = r[h];
    };
    auto xload = [&](int st, double (&r)[NB][4]) {
        const rsrc_t b = pf_rsrc(T + (size_t)(16 * st) * ldt);
#pragma unroll
        for (int u = 0; u < NB; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) r[u][q] = pf_ld(b, vx[u], 32 * q * ldt);
    };
    auto products = [&](int buf, const double (&r)[NB][4]) {
        const double *yb = Ys + buf * 16 * OB + lk * OB + pi;
        const double *xb = Ys + buf * 16 * OB + lk * OB + 16 * (wave & 3) + li;
        double v[2][4];
#pragma unroll
        for (int f = 0; f < 4; ++f) v[0][f] = yb[16 * f];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (q < 3) {
#pragma unroll
                for (int f = 0; f < 4; ++f) v[(q + 1) & 1][f] = yb[(q + 1) * 4 * OB + 16 * f];
            }
#pragma unroll
            for (int u = 0; u < NB; ++u)
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    const double x = DIAG ? xb[q * 4 * OB] : r[u][q];
                    if constexpr (LP) accf[u][f] = mfma_f32((float)v[q & 1][f], (float)x, accf[u][f]);
                    else acc[u][f] = mfma_f64(v[q & 1][f], x, acc[u][f]);
                }
            if constexpr (!LP && !DIAG) {
                /* one LDS read behind each of the first products */
                if (q < 3) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 4 * NB - 2, 0);
                }
            }
        }
    };
    if (S > 0) yload(0, y[0]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (!DIAG) xload(j, x[j]);
        else if (j <= wave && wave < nrb) xload(S + j, x[j]);
    }
    if (S > 0) {
#pragma unroll
        for (int j = 1; j < 4; ++j) yload(j, y[j]);
        ystore(0, y[0]);
        yload(4, y[0]);
        __syncthreads();
        for (int st = 0; st < S; st += 4) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                ystore((j & 1) ^ 1, y[(j + 1) & 3]);
                yload(st + j + 5, y[(j + 1) & 3]);
                products(j & 1, x[j]);
                if (!DIAG) xload(st + j + 4, x[j]);
                __syncthreads();
            }
        }
    }
    const int vt = (li + lk * ldt) * 8;
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        const int rb = rb0 + wave + NW * u;
        if (rb >= nrb) continue;
        v4d old[4];
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int s = 0; s < 4; ++s) old[f][s] = x[f][u][s] - (LP ? (double)accf[u][f][s] : acc[u][f][s]);
        if constexpr (DIAG) {
#pragma unroll
            for (int f = 0; f < 4; ++f)
                if (f <= rb) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) Db[pf_low(rb, f) + 64 * s + lane] = old[f][s];
                }
        } else {
            pf_subst(Db, lane, old);
            const rsrc_t t = pf_rsrc(T + C + 16 * rb + (size_t)C * ldt);
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int s = 0; s < 4; ++s) pf_st(old[f][s], t, vt, (16 * f + 4 * s) * ldt * 8);
        }
    }
}

template <int POTRF_WAVES, bool LP = false>
__global__ __launch_bounds__(POTRF_WAVES * 64, 2) void potrf_jobs_kernel(PotrfJobs J)
{
    constexpr int NW = POTRF_WAVES, NT = NW * 64;
    /* Ys holds the staged shared rows, Xs the 64 x 64 inverse on its way out,
     * Db the diagonal block's lower 16 x 16 blocks, which turn into L with the
     * inverses on the diagonal, and Ld the diagonal ones of L */
    __shared__ double Xs[OB * OB], Ys[2 * 16 * OB], Db[PF_LOW], Ld[4 * PF_BLK], Id[PF_BLK];
    __shared__ int s_fail, s_job;
    for (int e = threadIdx.x; e < PF_BLK; e += NT) Id[e] = (e & 15) == (e >> 4) ? 1.0 : 0.0;
    if (!J.batch && *J.info != 0) return;
    /* the single-job form is on the critical path of the factorisation:
     * its waves win issue arbitration against co-resident update waves */
    __builtin_amdgcn_s_setprio(2);
  for (int pass = 0;; ++pass) {
    if (threadIdx.x == 0) {
        s_job = J.queue ? atomicAdd(J.queue, 1) : (pass == 0 ? (int)blockIdx.x : J.count);
        s_fail = 0;
    }
    __syncthreads();
    const int job = __builtin_amdgcn_readfirstlane(s_job);
    if (job >= J.count) break;
    double *T = J.A + (J.off ? J.off[job] : 0);
    double *dinv = J.dinv + (J.doff ? J.doff[job] : 0);
    const int np = J.np ? J.np[job] : J.np0;
    const int ldt = J.ld ? J.ld[job] : (J.ld0 ? J.ld0 : np);
    const int nvalid = J.nvalid ? J.nvalid[job] : J.nvalid0;

    for (int C = 0; C < np; C += OB) {
        /* (kept from being taken out of the loop: the addresses formed from it
         * need more registers than there are) */
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lk = lane >> 4;
        const int W = min(OB, np - C), nfb = W >> 4;
        /* of a last block column narrower than 64 the blocks past the matrix hold
         * finite values; whatever is formed from them is masked */
        if (nfb < 4) {
            for (int e = tid; e < PF_LOW; e += NT) {
                const int b = e >> 8, i = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3;
                if (i >= nfb) Db[e] = (b == i * (i + 3) / 2 && (e & 15) == ((e >> 4) & 15)) ? 1.0 : 0.0;
            }
        }
        /* (a) for the diagonal block: of a first one, its values */
        jobs_update<NW, 1, LP, true>(T, ldt, C, 0, nfb, Ys, Db, tid);
        __syncthreads();
        /* (b), as in the panel's chain: wave 0 the columns, the others what
         * comes after them; wave 3 repeats the first block for its inverse
         * when the first step has no lane left for the identity */
#pragma unroll 1
        for (int cb = 0; cb < nfb; ++cb) {
            if (wave == 0 || (wave == 3 && cb == 1 && nfb == 4)) {
                const int c = wave == 0 ? cb : 0;
                const int fail = pf_step16(Db, Ld, Id, c, wave == 0 ? nfb - cb : 1, lane);
                if (lane == 0 && fail) s_fail = C + 16 * c + fail - 1 < nvalid ? C + 16 * c + fail : -1;
            } else if (cb > 0 && cb < 3 && wave < 3) {
                /* what step cb-1 takes off the columns after cb: (2,2), (3,2),
                 * (3,3), then (3,3) */
                for (int u = wave - 1; u < (cb == 1 ? 3 : 1); u += 2) {
                    const int i = u == 0 && cb == 1 ? 2 : 3, j = u == 2 || cb == 2 ? 3 : 2;
                    pf_take16(Db, i, j, cb - 1, lane);
                }
            }
            __syncthreads();
            if (s_fail) break;
            if (cb + 1 < nfb) {
                /* column cb+1 takes off step cb: block (cb + 1 + wave, cb + 1) */
                const int i = cb + 1 + wave;
                if (i < nfb) {
                    pf_take16(Db, i, cb + 1, cb, lane);
                }
                __syncthreads();
            }
        }
        if (s_fail) break;
        /* (c) inverse into dinv (zero past the matrix) and Xs, L into the matrix */
        pf_inverse<NT>(Db, Xs, dinv + (size_t)(C / OB) * OB * OB, W, tid, wave, lane);
        if (tid < 256) {
#pragma unroll
            for (int b = 0; b < 10; ++b) {
                const int i = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3, j = b - i * (i + 1) / 2;
                const double v = i == j ? Ld[j * PF_BLK + tid] : Db[b * PF_BLK + tid];
                if (i < nfb && (i > j || (tid & 15) >= (tid >> 4)))
                    T[(C + 16 * i + (tid & 15)) + (size_t)(C + 16 * j + (tid >> 4)) * ldt] = v;
            }
        }
        /* (a) and (d) for the rows below */
        {
            const int nrb = (np - C) >> 4;
            int rb0 = 4;
            for (; nrb - rb0 > NW; rb0 += 2 * NW) jobs_update<NW, 2, LP, false>(T, ldt, C, rb0, nrb, Ys, Db, tid);
            if (rb0 < nrb) jobs_update<NW, 1, LP, false>(T, ldt, C, rb0, nrb, Ys, Db, tid);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (J.batch) J.info[job] = s_fail > 0 ? s_fail : 0;
        else if (s_fail > 0) *J.info = J.iinfo + s_fail;
    }
    __syncthreads();
  }
}

void potrf_diag(double *Akk, int ldt, double *dinv, int iinfo, int nvalid, int *info, int waves, hipStream_t s)
{
    PotrfJobs J = {};
    J.A = Akk; J.dinv = dinv;
    J.np0 = ldt; J.ld0 = ldt; J.nvalid0 = nvalid;
    J.count = 1; J.info = info; J.iinfo = iinfo; J.batch = 0;
    if (waves == 8) hipLaunchKernelGGL(potrf_jobs_kernel<8>, dim3(1), dim3(512), 0, s, J);
    else hipLaunchKernelGGL(potrf_jobs_kernel<4>, dim3(1), dim3(256), 0, s, J);
}

/* Batched form: `count` matrices, job j of order np[j] (multiple of 16)
 * at A + off[j] with leading dimension ld[j] (null: np[j]), inverses at
 * dinv + doff[j]; info[j] = first failing column or 0.  `queue` is a
 * zeroed device counter; jobs are taken in index order by `grid`
 * persistent workgroups (grid <= 0: as many as are resident at once; sort
 * the jobs largest first for balance). */
template <int W, bool LP>
static int potrf_jobs_resident()
{
    static int resident = 0;
    if (!resident) {
        int dev = 0, ncu = 0, per = 0;
        CHX_HIP(hipGetDevice(&dev));
        CHX_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
        CHX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, potrf_jobs_kernel<W, LP>, W * 64, 0));
        resident = ncu * (per > 0 ? per : 1);
    }
    return resident;
}

template <int W, bool LP>
static void potrf_jobs_launch(const PotrfJobs &J, int grid, hipStream_t s)
{
    if (grid <= 0) grid = potrf_jobs_resident<W, LP>();
    if (grid > J.count) grid = J.count;
    hipLaunchKernelGGL((potrf_jobs_kernel<W, LP>), dim3(grid), dim3(W * 64), 0, s, J);
}

void potrf_jobs(double *A, const long long *off, const int *np, const int *ld, const int *nvalid, double *dinv,
                const long long *doff, int count, int *queue, int *info, int grid, hipStream_t s, int waves, bool lp)
{
    PotrfJobs J = {};
    J.A = A; J.off = off; J.np = np; J.ld = ld; J.nvalid = nvalid; J.dinv = dinv; J.doff = doff;
    J.count = count; J.queue = queue; J.info = info; J.batch = 1;
    if (count <= 0) return;
    if (waves == 8) {
        if (lp) potrf_jobs_launch<8, true>(J, grid, s);
        else potrf_jobs_launch<8, false>(J, grid, s);
    } else {
        if (lp) potrf_jobs_launch<4, true>(J, grid, s);
        else potrf_jobs_launch<4, false>(J, grid, s);
    }
}

void potrf_jobs_prepare()
{
    (void)potrf_jobs_resident<4, false>();
    (void)potrf_jobs_resident<8, false>();
    (void)potrf_jobs_resident<4, true>();
    (void)potrf_jobs_resident<8, true>();
}

} /* namespace k */
} /* namespace chx */
