/*
 * Direct cross-correlation kernel for gfx950 (the "plain" visibility path)
 * with a Gaussian or smearing factor per baseline; without one the sum is a
 * matrix product (xcorr_product.hip), but for few sources or stations.
 *
 * Computes, for every baseline (p > q) outside the uv filter,
 *     V_pq += sum_s smear_s(pq) * J_first(s) B_s J_second(s)^H
 * with first/second = (p, q) in the non-CASA convention and (q, p) in the
 * CASA convention (oskar/correlate/define_cross_correlate.h:34-77 and
 * oskar/correlate/src/oskar_cross_correlate_omp.cpp:33-156), and the scalar
 * (Stokes-I) form V_pq += sum_s smear_s I_s J_first conj(J_second)
 * (define_cross_correlate.h:113-155).
 *
 * Work decomposition (MI355X-specific, not the reference's):
 *  - A workgroup of 256 threads (four wave64s) owns a block of 32 "first"
 *    stations x 16 "second" stations.  Thread t owns first station t/8 and
 *    second stations t%8 and t%8 + 8.  In the matrix form M = J_first * B
 *    is formed once per (source, first station) of a staged tile, in LDS
 *    in place of J_first, and read by the 16 baselines that need it.
 *  - Only blocks that hold a baseline are launched, as one list of (split,
 *    block) items that the XCDs share evenly.
 *  - Sources are streamed in tiles of TILE sources.  The Jones values of the
 *    48 stations are loaded as 16-byte vectors, one station row of the tile
 *    per wave and instruction (64 lanes on consecutive bytes), and stored
 *    transposed in LDS as [source][vector][station], so the inner loop
 *    reads a first-station value that is broadcast to 8 lanes and
 *    consecutive second-station vectors, without bank conflicts.  Source
 *    parameters are stored as 4-value vectors, one LDS read each.
 *  - The factors of a baseline and source: the Gaussian only for sources
 *    that are extended (a wave's sources are the same), the smearing by the
 *    polynomials of Sinc (device_common.h).  The second-station Jones is
 *    scaled by their product, and every term of M J^H is one fused
 *    multiply-add into the tile sum.
 *  - Single precision: each tile is summed in FP32 registers, then folded
 *    into FP64 accumulators (cross-tile sums in FP64).  Double precision
 *    accumulates in FP64 throughout.
 *  - The source range is split over workgroups; partial sums go to an FP64
 *    workspace and a second kernel adds them to vis in a fixed order.  No
 *    atomics are used, so results are identical from run to run.
 *
 * Bound: vector instructions.  FP32 matrices with all factors take 82 per
 * evaluation, 40 of them the contraction (163 with library sines, divisions
 * and both sinc branches, 92 with the sinc's last form past MID), and the
 * vector unit is busy throughout: 512 stations x 20,000 sources 10.8 ->
 * 5.2 ms (5.73 without the form up to WIDE).  FP64 with both smearings
 * takes 82 (565), vector unit 74 % busy at three waves per SIMD: 255 x
 * 10,007 sources 4.62 -> 1.20 ms.  Scalars with bandwidth smearing in FP32,
 * 351 x 50,001: 2.52 -> 1.37 ms (1.43 with the flux in an LDS
 * read of its own: LDS was active 71 % of the time).
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "device_common.h"
#include "private.h"
#include "workspace.h"
#include "xcorr_common.h"

using namespace oskar_amd;

namespace {

constexpr int BLOCK_A = 32;    /* "first" stations per workgroup */
constexpr int BLOCK_B = 16;    /* "second" stations per workgroup */
constexpr int THREADS = 256;

/* exp2 of a Gaussian's exponent, whose a, b, c carry -log2(e) (FP32: the
 * hardware's exp2), or exp of it with a, b, c negated (FP64). */
__device__ __forceinline__ float gauss_scale(float) { return -1.44269504f; }
__device__ __forceinline__ double gauss_scale(double) { return -1.0; }
__device__ __forceinline__ float gauss_exp(float x)
{
    return __builtin_amdgcn_exp2f(x);
}
__device__ __forceinline__ double gauss_exp(double x) { return exp(x); }

/* The smearing factors of a thread's two baselines for one source, times
 * the Gaussian factors already in sm.  The sinc form is chosen by the
 * largest argument in the wave: long baselines and sources far from the
 * phase centre take the wider forms. */
template <typename FP, bool BS, bool TS>
__device__ __forceinline__ void smear_factors(
        const BaselineTerms<FP, TS> (&t)[2], FP l, FP m, FP n1, FP (&sm)[2])
{
    using S = Sinc<FP>;
    FP xb[2], xt[2], most = (FP) 0;
#pragma unroll
    for (int k = 0; k < 2; ++k)
    {
        if (BS)
        {
            xb[k] = t[k].uu * l + t[k].vv * m + t[k].ww * n1;
            most = fmax(most, fabs(xb[k]));
        }
        if (TS)
        {
            xt[k] = t[k].du * l + t[k].dv * m + t[k].dw * n1;
            most = fmax(most, fabs(xt[k]));
        }
    }
    auto apply = [&](auto f) __attribute__((always_inline))
    {
#pragma unroll
        for (int k = 0; k < 2; ++k)
        {
            if (BS) sm[k] *= f(xb[k]);
            if (TS) sm[k] *= f(xt[k]);
        }
    };
    if (!__any(most > S::SMALL))
        apply([](FP x) { return S::small(x); });
    else if (!__any(most > S::MID))
        apply([](FP x) { return S::mid(x); });
    else if (!__any(most > S::WIDE))
        apply([](FP x) { return S::wide(x); });
    else
        apply([](FP x) { return S::large(x); });
}

/* Number of reals per Jones value and the source-tile length.  A Jones
 * value is moved as VPE vectors of VR reals (16 bytes, or 8 for a float
 * complex scalar); TILE * VPE = 64, so one wave loads one station row of
 * a tile with consecutive lanes on consecutive bytes. */
/* Matrix kernels stage 16 sources per tile: with one source per iteration
 * of the inner loop every FP32 matrix variant fits 128 VGPRs and 26 KB of
 * LDS, four waves per SIMD. */
template <typename FP, bool MATRIX> struct Geometry
{
    static constexpr int NR = MATRIX ? 8 : 2;
    static constexpr int TILE = MATRIX ? 16 : 64;
    static constexpr int VPE = MATRIX ? (sizeof(FP) == 4 ? 2 : 4) : 1;
    static constexpr int VR = NR / VPE;
    /* Fewest sources of a split (the inner loop's granularity). */
    static constexpr int LEAST = sizeof(FP) == 8 ? 4 : TILE;
    /* Station rows of a tile moved by one wave instruction. */
    static constexpr int RPI = 64 / (TILE * VPE);
    static_assert(RPI * TILE * VPE == 64, "whole station rows per wave");
};

/* Four source values, read from LDS as one vector. */
template <typename FP> struct alignas(4 * sizeof(FP)) Quad
{
    FP x, y, z, w;
};

/* The station blocks that hold a baseline with the required index order:
 * for first block ia (stations 32 ia ..), second blocks *ib0 .. *ib0 +
 * count - 1 (stations 16 ib ..). */
__host__ __device__ inline int blocks_in_row(int N, bool casa, int ia,
        int* ib0)
{
    const int a0 = ia * BLOCK_A;
    const int a_last = (a0 + BLOCK_A < N ? a0 + BLOCK_A : N) - 1;
    if (casa)
    {
        /* first < second */
        *ib0 = a0 / BLOCK_B;
        return a0 < N - 1 ? (N + BLOCK_B - 1) / BLOCK_B - *ib0 : 0;
    }
    /* first > second */
    *ib0 = 0;
    return a_last > 0 ? (a_last - 1) / BLOCK_B + 1 : 0;
}

/* Blocks of the rows before row ia: of every row but the last, 2 ia + 2, or
 * in the CASA order the whole row's blocks less 2 ia. */
__host__ __device__ inline int blocks_before(int N, bool casa, int ia)
{
    const int row = (N + BLOCK_B - 1) / BLOCK_B;
    return casa ? ia * (row + 1 - ia) : ia * (ia + 1);
}

/* The row of a block of the list, by the root of blocks_before(), whose
 * rounding is put right (a search row by row took 20 us of scalar code per
 * workgroup at 3000 stations). */
__host__ __device__ inline int block_row(int N, bool casa, int block)
{
    const float row = (float) ((N + BLOCK_B - 1) / BLOCK_B + 1);
    int ia = casa ? (int) (0.5f * (row - sqrtf(fmaxf(row * row -
            4.0f * (float) block, 0.0f)))) :
            (int) (0.5f * (sqrtf(4.0f * (float) block + 1.0f) - 1.0f));
#if defined(__HIP_DEVICE_COMPILE__)
    ia = __builtin_amdgcn_readfirstlane(ia);
#endif
    while (ia > 0 && blocks_before(N, casa, ia) > block) --ia;
    while (blocks_before(N, casa, ia + 1) <= block) ++ia;
    return ia;
}

/* FP64 matrices without the Gaussian factor fit three waves per SIMD (168
 * VGPRs and 52 KB of LDS: 1.25 -> 1.19 ms for 255 stations x 10,007
 * sources); with it they would spill (30 x 277 sources: 21.7 -> 24.6 us). */
template <typename FP, bool MATRIX, bool GAUSS, bool BS, bool TS>
__global__ __launch_bounds__(THREADS, MATRIX && !GAUSS && sizeof(FP) == 8 ?
        3 : 1)
void xcorr_direct_kernel(XcorrArgs<FP> A, int blocks)
{
    using G = Geometry<FP, MATRIX>;
    constexpr int NR = G::NR;
    constexpr int TILE = G::TILE;
    constexpr int VPE = G::VPE;
    constexpr int VR = G::VR;
    using V = Vec<FP, VR>;
    /* A station's value as vectors in planes of their own, so that lanes on
     * consecutive stations read consecutive vectors; the odd number of
     * stations per plane spreads the transposed stores over banks. */
    __shared__ V sJa[TILE][VPE][BLOCK_A + 1];
    __shared__ V sJb[TILE][VPE][BLOCK_B + 1];
    __shared__ Quad<FP> sFlux[TILE];      /* I, Q, U, V */
    __shared__ Quad<FP> sDir[TILE];       /* l, m, n - 1, I */
    __shared__ Quad<FP> sExt[TILE];       /* a, b, c */

    const int N = A.num_stations;
    /* Workgroup w runs on XCD w % 8; each XCD takes a contiguous range of
     * (split, block) items, so that all have the same work (with a grid of
     * all blocks, XCDs held whole block rows: 2x the average on 255
     * stations) and the blocks of a split share an L2. */
    const int total = (int) gridDim.x, wg = (int) blockIdx.x;
    const int xq = total / 8, xr = total % 8, xcd = wg % 8;
    const int item = xcd * xq + min(xcd, xr) + wg / 8;
    const int split = item / blocks;
    const bool casa = A.use_casa != 0;
    const int block = item % blocks, ia = block_row(N, casa, block);
    const int a0 = ia * BLOCK_A;
    const int b0 = (block - blocks_before(N, casa, ia)) * BLOCK_B +
            (casa ? a0 : 0);
    const int tid = threadIdx.x;
    const int la = tid >> 3;
    /* Second stations lb and lb + 8: the eight lanes of a wave that share
     * a first station read eight consecutive second stations, which fall
     * in distinct LDS banks. */
    const int lb = tid & 7;
    const int sa = a0 + la;
    const int sb[2] = { b0 + lb, b0 + lb + 8 };

    /* Baseline terms and validity for the two baselines of this thread:
     * in[k] = a real baseline in this block, ok[k] = also inside the uv
     * filter.  With split sources every real baseline writes its partial
     * sum and the reduction alone applies the filter. */
    BaselineTerms<FP, TS> bt[2];
    bool ok[2], in[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
    {
        in[k] = sa < N && sb[k] < N &&
                (A.use_casa ? (sa < sb[k]) : (sa > sb[k]));
        /* Out-of-range slots use the dummy pair (1, 0); N >= 2 here. */
        const int sp = in[k] ? max(sa, sb[k]) : 1;
        const int sq = in[k] ? min(sa, sb[k]) : 0;
        bt[k].init(A, sp, sq);
        ok[k] = in[k] &&
                !(bt[k].uv_len < A.uv_min || bt[k].uv_len > A.uv_max);
    }

    const int s_begin = split * A.src_per_split;
    const int s_end = min(A.num_sources, s_begin + A.src_per_split);

    double acc[2][NR];
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < NR; ++r) acc[k][r] = 0.0;

    const FP* J = (const FP*) A.jones;
    /* Tile loads: instruction i of wave w moves station rows
     * (w + 4 i) RPI + r, r < RPI, of the block (rows 0-31 first stations,
     * 32-47 second stations); lane (r, s, q) moves vector q of source s of
     * row r.  Whole-vector loads need the Jones array aligned to a vector,
     * which element-aligned arrays are; otherwise the same mapping moves
     * one real at a time. */
    constexpr int RPI = G::RPI;
    const int lane = tid & 63, wave = tid >> 6;
    const int lq = lane % VPE, ls = (lane / VPE) % TILE;
    const int lr = lane / (TILE * VPE);
    const bool vec_ok = (((uintptr_t) J) % sizeof(V)) == 0;
    for (int s0 = s_begin; s0 < s_end; s0 += TILE)
    {
        const int ns = min(TILE, s_end - s0);
        __syncthreads();
        const bool s_ok = ls < ns;
#pragma unroll
        for (int i = 0; i < (BLOCK_A + BLOCK_B) / (4 * RPI); ++i)
        {
            const int st = (wave + 4 * i) * RPI + lr;
            const bool first = st < BLOCK_A;
            const int station = first ? a0 + st : b0 + (st - BLOCK_A);
            V* dst = first ? &sJa[ls][lq][st] : &sJb[ls][lq][st - BLOCK_A];
            const FP* src = J + ((size_t) station * A.num_sources + s0 +
                    ls) * NR + lq * VR;
            V x;
#pragma unroll
            for (int r = 0; r < VR; ++r) x.v[r] = (FP) 0;
            if (station < N && s_ok)
            {
                if (vec_ok)
                    x = *(const V*) src;
                else
                {
#pragma unroll
                    for (int r = 0; r < VR; ++r) x.v[r] = src[r];
                }
            }
            *dst = x;
        }
        for (int s = tid; s < TILE; s += THREADS)
        {
            const bool in = s < ns;
            const int g = s0 + s;
            const FP z = (FP) 0;
            sFlux[s] = Quad<FP>{in ? A.I[g] : z,
                    (MATRIX && in) ? A.Q[g] : z,
                    (MATRIX && in) ? A.U[g] : z,
                    (MATRIX && in) ? A.V[g] : z};
            if (BS || TS)
                sDir[s] = Quad<FP>{in ? A.l[g] : z, in ? A.m[g] : z,
                        in ? A.n[g] - (FP) 1 : z, in ? A.I[g] : z};
            if (GAUSS)
            {
                /* .w: whether the source is extended. */
                const FP f = gauss_scale(z);
                const FP ea = in ? A.a[g] : z, eb = in ? A.b[g] : z;
                const FP ec = in ? A.c[g] : z;
                sExt[s] = Quad<FP>{f * ea, f * eb, f * ec,
                        (FP) (ea != z || eb != z || ec != z)};
            }
        }
        __syncthreads();
        if constexpr (MATRIX)
        {
            /* M = J_first * B once per (source, first station) of the tile,
             * in place of J_first.  Each entry is read and written by one
             * thread. */
            for (int i = tid; i < TILE * BLOCK_A; i += THREADS)
            {
                const int s = i / BLOCK_A, a = i % BLOCK_A;
                const Quad<FP> fl = sFlux[s];
                FP ja[8], M[8];
#pragma unroll
                for (int r = 0; r < 8; ++r)
                    ja[r] = sJa[s][r / VR][a].v[r % VR];
                row_times_brightness<FP>(ja, fl.x, fl.y, fl.z, fl.w, M);
                row_times_brightness<FP>(ja + 4, fl.x, fl.y, fl.z, fl.w,
                        M + 4);
#pragma unroll
                for (int v = 0; v < VPE; ++v)
                {
                    V x;
#pragma unroll
                    for (int r = 0; r < VR; ++r) x.v[r] = M[v * VR + r];
                    sJa[s][v][a] = x;
                }
            }
            __syncthreads();
        }

        FP t[2][NR];
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int r = 0; r < NR; ++r) t[k][r] = (FP) 0;

        /* The extended sources of the tile, one bit each: a branch per source
         * that waits for no LDS read. */
        uint64_t extended = 0;
        if (GAUSS)
        {
            static_assert(TILE <= 64, "a bit per source");
            extended = __ballot(lane < TILE && sExt[lane % TILE].w != (FP) 0);
        }
        /* Two sources per iteration in the FP32 scalar form; one in the
         * matrix form (more registers would leave three waves per SIMD)
         * and in FP64. */
        constexpr int UNROLL = (sizeof(FP) == 4 && !MATRIX) ? 2 : 1;
        /* Past ns: zeros (FP32 runs over them: with a count that varies the
         * matrix kernels pass 128 VGPRs). */
        const int count = G::LEAST < TILE ? ns : TILE;
#pragma unroll UNROLL
        for (int s = 0; s < count; ++s)
        {
            /* Scalars: the flux, with the direction where that is read. */
            FP flux = (BS || TS) ? (FP) 0 : sFlux[s].x;
            FP sm[2] = {(FP) 1, (FP) 1};
            if (GAUSS)
            {
                if (extended >> s & 1u)
                {
                    const Quad<FP> e = sExt[s];
#pragma unroll
                    for (int k = 0; k < 2; ++k)
                        sm[k] = gauss_exp(e.x * bt[k].uu2 +
                                e.y * bt[k].uuvv + e.z * bt[k].vv2);
                }
            }
            if (BS || TS)
            {
                const Quad<FP> d = sDir[s];
                flux = d.w;
                smear_factors<FP, BS, TS>(bt, d.x, d.y, d.z, sm);
            }
            /* The values of this thread's stations. */
            auto get = [](const V* planes, int pitch, FP* x)
            {
#pragma unroll
                for (int v = 0; v < VPE; ++v)
                {
                    const V y = planes[v * pitch];
#pragma unroll
                    for (int r = 0; r < VR; ++r) x[v * VR + r] = y.v[r];
                }
            };
            FP ja[NR];
            get(&sJa[s][0][la], BLOCK_A + 1, ja);
            if (MATRIX)
            {
                /* The tile holds M = J_first * B (formed after staging). */
                const FP* M = ja;
#pragma unroll
                for (int k = 0; k < 2; ++k)
                {
                    /* t += smear * M * J_second^H (define_multiply.h:54-67):
                     * (M J^H).a = M.a conj(J.a) + M.b conj(J.b), etc.  The
                     * smearing factor scales J_second; each term is one
                     * fused multiply-add into the tile sum. */
                    FP jb[8], w[8];
                    get(&sJb[s][0][lb + 8 * k], BLOCK_B + 1, jb);
#pragma unroll
                    for (int r = 0; r < 8; ++r)
                        w[r] = jb[r] * sm[k];
                    FP* T = t[k];
                    T[0] += M[0] * w[0]; T[0] += M[1] * w[1];
                    T[0] += M[2] * w[2]; T[0] += M[3] * w[3];
                    T[1] += M[1] * w[0]; T[1] -= M[0] * w[1];
                    T[1] += M[3] * w[2]; T[1] -= M[2] * w[3];
                    T[2] += M[0] * w[4]; T[2] += M[1] * w[5];
                    T[2] += M[2] * w[6]; T[2] += M[3] * w[7];
                    T[3] += M[1] * w[4]; T[3] -= M[0] * w[5];
                    T[3] += M[3] * w[6]; T[3] -= M[2] * w[7];
                    T[4] += M[4] * w[0]; T[4] += M[5] * w[1];
                    T[4] += M[6] * w[2]; T[4] += M[7] * w[3];
                    T[5] += M[5] * w[0]; T[5] -= M[4] * w[1];
                    T[5] += M[7] * w[2]; T[5] -= M[6] * w[3];
                    T[6] += M[4] * w[4]; T[6] += M[5] * w[5];
                    T[6] += M[6] * w[6]; T[6] += M[7] * w[7];
                    T[7] += M[5] * w[4]; T[7] -= M[4] * w[5];
                    T[7] += M[7] * w[6]; T[7] -= M[6] * w[7];
                }
            }
            else
            {
#pragma unroll
                for (int k = 0; k < 2; ++k)
                {
                    FP jb[2];
                    get(&sJb[s][0][lb + 8 * k], BLOCK_B + 1, jb);
                    /* J_first * conj(J_second) * (smear * I) */
                    const FP w = sm[k] * flux;
                    const FP re = ja[0] * jb[0] + ja[1] * jb[1];
                    const FP im = ja[1] * jb[0] - ja[0] * jb[1];
                    t[k][0] += re * w;
                    t[k][1] += im * w;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int r = 0; r < NR; ++r) acc[k][r] += (double) t[k][r];
    }

    /* Output: direct accumulation into vis, or per-split partials. */
#pragma unroll
    for (int k = 0; k < 2; ++k)
    {
        if (!(A.num_splits == 1 ? ok[k] : in[k])) continue;
        const int sp = max(sa, sb[k]), sq = min(sa, sb[k]);
        const int bl = sq * (N - 1) - (sq - 1) * sq / 2 + sp - sq - 1;
        if (A.num_splits == 1)
        {
            FP* v = (FP*) A.vis + (size_t) (A.offset_out + bl) * NR;
#pragma unroll
            for (int r = 0; r < NR; ++r) v[r] += (FP) acc[k][r];
        }
        else
        {
            const size_t nb = (size_t) N * (N - 1) / 2;
            double* w = A.partial + ((size_t) split * nb + bl) * NR;
#pragma unroll
            for (int r = 0; r < NR; ++r) w[r] = acc[k][r];
        }
    }
}

/* Adds the split partial sums to vis in a fixed order, skipping baselines
 * outside the uv filter.  Grid: y = the lower station index q, x over the
 * consecutive reals of its baselines (p, q).  GROUPS groups of a workgroup
 * add a share of the splits each (consecutive threads on consecutive
 * partials), and the shares are added in order: 4 where there are many
 * splits, so that a small array's sums are not one long chain (60 stations,
 * 205 splits: 66 us with a thread per baseline). */
template <typename FP, int NR, int GROUPS>
__global__ __launch_bounds__(256)
void xcorr_reduce_kernel(XcorrArgs<FP> A)
{
    constexpr int VALUES = 256 / GROUPS;
    __shared__ double sums[GROUPS > 1 ? GROUPS - 1 : 1][VALUES];
    const int N = A.num_stations;
    const size_t nb = (size_t) N * (N - 1) / 2;
    const int q = blockIdx.y;
    const int at = threadIdx.x % VALUES, group = threadIdx.x / VALUES;
    const int e = blockIdx.x * VALUES + at;
    const int count = (N - 1 - q) * NR;
    if ((int) blockIdx.x * VALUES >= count) return;
    const size_t first = (size_t) baseline_index(N, q + 1, q) * NR;
    double sum = 0.0;
    if (e < count)
    {
        const int per = (A.num_splits + GROUPS - 1) / GROUPS;
        const int k1 = min(A.num_splits, (group + 1) * per);
        const double* w = A.partial + first + e;
#pragma unroll 4
        for (int k = group * per; k < k1; ++k) sum += w[k * nb * NR];
    }
    if (GROUPS > 1)
    {
        if (group > 0) sums[group - 1][at] = sum;
        __syncthreads();
        if (group > 0) return;
#pragma unroll
        for (int g = 0; g < GROUPS - 1; ++g) sum += sums[g][at];
    }
    if (e >= count) return;
    BaselineTerms<FP, false> t;
    t.init(A, q + 1 + e / NR, q);
    if (t.uv_len < A.uv_min || t.uv_len > A.uv_max) return;
    FP* v = (FP*) A.vis + (size_t) A.offset_out * NR + first + e;
    *v += (FP) sum;
}

/* FP64 workspace for the split partial sums, one per (device, stream),
 * grown on demand and kept for the life of the process. */
void* workspace_get(size_t bytes, hipStream_t stream, hipError_t* err)
{
    int dev = 0;
    *err = hipGetDevice(&dev);
    if (*err != hipSuccess) return nullptr;
    return ws_acquire(WS_XCORR_SPLIT, dev, stream, bytes, err);
}

/* fixed: the device's scratch array (allocation-free entry point); NULL:
 * the per-stream workspace. */
template <typename FP, bool MATRIX, bool GAUSS, bool BS, bool TS>
hipError_t launch_t(XcorrArgs<FP> A, hipStream_t stream, double* fixed)
{
    using G = Geometry<FP, MATRIX>;
    const int N = A.num_stations;
    const int na = (N + BLOCK_A - 1) / BLOCK_A;
    int blocks = 0, ib0 = 0;
    for (int ia = 0; ia < na; ++ia)
        blocks += blocks_in_row(N, A.use_casa != 0, ia, &ib0);
    if (blocks == 0 || A.num_sources <= 0) return hipSuccess;
    /* Splits: about 12 rounds of four workgroups per CU, so that the last
     * round's idle time is small, with at least 8 tiles of sources each
     * (the prologue and the partial sums cost about one).  Where that leaves
     * the chip idle, more while there is less than a round, down to LEAST
     * sources each (30 stations x 277 sources in FP64: 8 workgroups of four
     * tiles 80 us, 36 of one 21.6 us, 140 of 4 sources 17.7 us), as long as a
     * split saves more than its partial sums cost: going from k - 1 to k
     * saves `each` us per source / (k (k - 1)), a split's sums take their
     * bytes at 1.1 TB/s (written scattered and read again), and the second
     * kernel 3 us (512 x 20 FP32 matrices: 22 us as one split, 36 as two; 300
     * x 32 FP64: 25, 23 as two, 36 as eight; 512 x 32: 32 and 50 as three). */
    constexpr double each = GAUSS || BS || TS ?
            (MATRIX ? (sizeof(FP) == 8 ? 0.65 : 0.43) :
            (sizeof(FP) == 8 ? 0.25 : 0.14)) :
            (MATRIX ? (sizeof(FP) == 8 ? 0.45 : 0.3) :
            (sizeof(FP) == 8 ? 0.1 : 0.08));
    constexpr int round = MATRIX && sizeof(FP) == 8 ? 768 : 1024;
    const size_t nb = (size_t) N * (N - 1) / 2;
    const double sums = nb * G::NR * sizeof(double) / 1.1e6;
    const double saved = each * A.num_sources;
    int few = saved > 2.0 * (3.0 + 2.0 * sums) ?
            (int) (0.5 + sqrt(saved / sums + 0.25)) : 1;
    /* Whole units of LEAST sources, the nearest number per split. */
    const int units = (A.num_sources + G::LEAST - 1) / G::LEAST;
    const int unit_split = max(1, (2 * units + few) / (2 * few));
    few = min((units + unit_split - 1) / unit_split, round / blocks);
    int splits = (12 * 1024 + blocks - 1) / blocks;
    const int max_splits = max(1, max(A.num_sources / (8 * G::TILE), few));
    splits = max(1, min(splits, min(max_splits, 256)));
    /* One split writes vis directly and needs no partial sums. */
    splits = max(1, (int) min((size_t) splits,
            XCORR_PARTIAL_BYTES / (nb * G::NR * sizeof(double))));
    int per = (A.num_sources + splits - 1) / splits;
    const int unit = per < G::TILE ? G::LEAST : G::TILE;
    per = ((per + unit - 1) / unit) * unit;
    splits = (A.num_sources + per - 1) / per;
    A.src_per_split = per;
    A.num_splits = splits;
    A.partial = nullptr;
    if (splits > 1 && fixed) A.partial = fixed;
    else if (splits > 1)
    {
        hipError_t err = hipSuccess;
        A.partial = (double*) workspace_get(
                (size_t) splits * nb * G::NR * sizeof(double), stream, &err);
        if (err != hipSuccess) return err;
    }
    hipLaunchKernelGGL((xcorr_direct_kernel<FP, MATRIX, GAUSS, BS, TS>),
            dim3((unsigned) blocks * (unsigned) splits), dim3(THREADS), 0,
            stream, A, blocks);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess || splits == 1) return err;
    const int reals = (N - 1) * G::NR;
    if (splits >= 16)
        hipLaunchKernelGGL((xcorr_reduce_kernel<FP, G::NR, 4>),
                dim3((unsigned) ((reals + 63) / 64), (unsigned) (N - 1)),
                dim3(256), 0, stream, A);
    else
        hipLaunchKernelGGL((xcorr_reduce_kernel<FP, G::NR, 1>),
                dim3((unsigned) ((reals + 255) / 256), (unsigned) (N - 1)),
                dim3(256), 0, stream, A);
    return hipGetLastError();
}

/* Whether the per-baseline kernel is done with few sources or stations sooner
 * than the product, whose workgroups are few (64 x 64 stations of scalars each)
 * and take long stages.  Product -> per baseline, us, FP32: scalars 200 stations x 16 sources
 * 17.6 -> 12, 512 x 64 21 -> 12.5, 512 x 128 21 -> 18.5, 1000 x 64 23 -> 19
 * (but 700 x 96 23 -> 22 and 1100 x 64 24 -> 24); matrices 200 x 16 17 -> 12,
 * 300 x 32 20 -> 17, 3000 x 16 175 -> 124 (but 1100 x 24 51 -> 50, 200 x 48
 * 19 -> 19).  Arrays of up to 32 stations of scalars are a corner of one of its
 * tiles: 2 x 100,000 FP32 58 -> 39, FP64 72 -> 47, 32 x 30,000 35 -> 26 and 47
 * -> 29 (but 32 x 100,000 53 -> 57, 64 x 10,000 24 -> 24). */
template <bool MATRIX> bool is_few(int num_sources, int num_stations)
{
    if (MATRIX)
        return num_sources <= 16 || (num_sources <= 32 && num_stations <= 512);
    return (num_sources <= 64 && num_stations <= 1024) ||
            (num_sources <= 128 && num_stations <= 512) ||
            (num_sources <= 65536 && num_stations <= 32) ||
            (num_sources <= 131072 && num_stations <= 16);
}

template <typename FP, bool MATRIX>
hipError_t dispatch(const XcorrArgs<FP>& A, bool gauss, bool bs, bool ts,
        hipStream_t s, double* fixed)
{
    /* No factor depends on the baseline: one matrix product, but for few
     * sources or stations. */
    if (!gauss && !bs && !ts && !is_few<MATRIX>(A.num_sources,
            A.num_stations))
        return xcorr_product_launch<FP, MATRIX>(A, s, fixed);
#define XC_CASE(G_, B_, T_) if (gauss == G_ && bs == B_ && ts == T_) \
        return launch_t<FP, MATRIX, G_, B_, T_>(A, s, fixed);
    XC_CASE(false, false, false) XC_CASE(false, false, true)
    XC_CASE(false, true, false)  XC_CASE(false, true, true)
    XC_CASE(true, false, false)  XC_CASE(true, false, true)
    XC_CASE(true, true, false)   XC_CASE(true, true, true)
#undef XC_CASE
    return hipErrorInvalidValue;
}

template <typename FP>
hipError_t build_and_launch(int matrix, const oskar_XcorrParams* p,
        const void* jones, const void* I, const void* Q, const void* U,
        const void* V, const void* l, const void* m, const void* n,
        const void* a, const void* b, const void* c, const void* st_u,
        const void* st_v, const void* st_w, const void* st_x,
        const void* st_y, void* vis, hipStream_t stream, bool no_alloc)
{
    XcorrArgs<FP> A;
    A.num_sources = p->num_sources;
    A.num_stations = p->num_stations;
    A.offset_out = p->offset_out;
    A.use_casa = p->use_casa;
    A.src_per_split = 0;
    A.num_splits = 1;
    A.jones = jones;
    A.I = (const FP*) I; A.Q = (const FP*) Q;
    A.U = (const FP*) U; A.V = (const FP*) V;
    A.l = (const FP*) l; A.m = (const FP*) m; A.n = (const FP*) n;
    A.a = (const FP*) a; A.b = (const FP*) b; A.c = (const FP*) c;
    A.st_u = (const FP*) st_u; A.st_v = (const FP*) st_v;
    A.st_w = (const FP*) st_w;
    A.st_x = (const FP*) st_x; A.st_y = (const FP*) st_y;
    A.uv_min = (FP) p->uv_min_lambda;
    A.uv_max = (FP) p->uv_max_lambda;
    A.inv_wl = (FP) p->inv_wavelength;
    A.frac_bw = (FP) p->frac_bandwidth;
    A.time_int = (FP) p->time_int_sec;
    const double ha = (double) (FP) p->gha0_rad;
    const double dec = (double) (FP) p->dec0_rad;
    A.sin_ha = (FP) sin(ha);
    A.cos_ha = (FP) cos(ha);
    A.sin_dec = (FP) sin(dec);
    A.cos_dec = (FP) cos(dec);
    A.vis = vis;
    A.partial = nullptr;
    if (A.num_stations < 2) return hipSuccess;
    double* fixed = nullptr;
    if (no_alloc)
    {
        const hipError_t err = xcorr_scratch(&fixed);
        if (err != hipSuccess) return err;
    }
    if (matrix)
        return dispatch<FP, true>(A, p->gaussian != 0,
                p->bandwidth_smearing != 0, p->time_smearing != 0, stream,
                fixed);
    return dispatch<FP, false>(A, p->gaussian != 0,
            p->bandwidth_smearing != 0, p->time_smearing != 0, stream, fixed);
}

} /* namespace */

extern "C" int oskar_amd_xcorr_launch(int precision, int matrix,
        const oskar_XcorrParams* p, const void* jones,
        const void* I, const void* Q, const void* U, const void* V,
        const void* l, const void* m, const void* n,
        const void* a, const void* b, const void* c,
        const void* st_u, const void* st_v, const void* st_w,
        const void* st_x, const void* st_y, void* vis, void* stream)
{
    if (precision == OSKAR_DOUBLE)
        return (int) build_and_launch<double>(matrix, p, jones, I, Q, U, V,
                l, m, n, a, b, c, st_u, st_v, st_w, st_x, st_y, vis,
                (hipStream_t) stream, false);
    return (int) build_and_launch<float>(matrix, p, jones, I, Q, U, V,
            l, m, n, a, b, c, st_u, st_v, st_w, st_x, st_y, vis,
            (hipStream_t) stream, false);
}

extern "C" int oskar_amd_xcorr_launch_no_alloc(int precision, int matrix,
        const oskar_XcorrParams* p, const void* jones,
        const void* I, const void* Q, const void* U, const void* V,
        const void* l, const void* m, const void* n,
        const void* a, const void* b, const void* c,
        const void* st_u, const void* st_v, const void* st_w,
        const void* st_x, const void* st_y, void* vis, void* stream)
{
    if (precision == OSKAR_DOUBLE)
        return (int) build_and_launch<double>(matrix, p, jones, I, Q, U, V,
                l, m, n, a, b, c, st_u, st_v, st_w, st_x, st_y, vis,
                (hipStream_t) stream, true);
    return (int) build_and_launch<float>(matrix, p, jones, I, Q, U, V,
            l, m, n, a, b, c, st_u, st_v, st_w, st_x, st_y, vis,
            (hipStream_t) stream, true);
}
