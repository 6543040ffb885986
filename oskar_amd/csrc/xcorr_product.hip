/*
 * The direct correlator for point sources without smearing, on the matrix
 * cores in the precision of the data (gfx950).
 *
 * Without a factor that depends on the baseline, the sum of
 * xcorr_direct.hip,
 *     V_pq = sum_s J_p(s) B_s J_q(s)^H   (p > q),
 * is one product V = M J^H with M = J B: rows (station, i), columns
 * (station, k), contracted over (source, j).  Scalar Jones values drop i, j
 * and k.  In real form, with X = [Re, Im] and Y = [Im, -Re] interleaved
 * along the contraction,
 *     Re V = X_M X_J^T,   Im V = Y_M X_J^T.
 * The CASA convention is the conjugate transpose of the same 2x2 block
 * (B is Hermitian).
 *
 * Instructions: v_mfma_f64_16x16x4 and v_mfma_f32_16x16x4, whose 4
 * contraction steps are one source of 2x2 matrices (j, Re/Im) or two
 * sources of scalars.  FP32 operands stay FP32 (no 16-bit split) and a
 * stage of sources (16 matrices or 32 scalars) is summed in FP32, then
 * added to FP64 accumulators, as the per-baseline kernels do.
 *
 * Tiles: a workgroup of four waves owns 64 x 64 rows (32 x 32 stations of
 * matrices, 64 x 64 of scalars), each wave 32 x 32 rows as 2 x 2 blocks of
 * Re and Im.  A wave whose stations hold no p > q pair issues no MFMA (its
 * SIMD serves the other workgroup of the CU), and on the diagonal the block
 * above it is skipped, so the padding is that of 16-station blocks.
 * Sources are staged through LDS (double-buffered, 33 KB per stage: two
 * workgroups per CU): a thread loads whole operand rows of a k-step (one row
 * of a station's matrix, consecutive threads on consecutive addresses,
 * prefetched in registers one stage ahead), forms the row of M for the
 * first side and writes the four contraction steps as [k-step][16-row
 * block][4][16], which an MFMA operand reads as 64 consecutive values.
 * K-steps come in pairs, one of real and one of imaginary parts, so that
 * the operands of Y are those of X with the two k-steps exchanged and the
 * sign of one taken by the instruction (FP64) or flipped (FP32): a third
 * fewer LDS reads and half or none of the flips of k-steps that hold both
 * parts (7.54 -> 7.36 ms and 0.87 -> 0.85 ms at the sizes below).
 *
 * Bound and measurements: the FP32 and FP64 MFMAs run on the multipliers of
 * the vector unit (no vector instruction issues beside them: matrix and
 * vector cycles add up to the kernel's time), so what counts beside the
 * MFMAs is the number of vector instructions of a stage, and the loads:
 * whole rows of the Jones array per wave instruction (8-byte loads 64 bytes
 * apart cost 13.8 ms instead of 8.1 in FP32).  The per-baseline kernel it
 * replaces read 48 bytes of LDS per evaluation and took, for 512 stations
 * x 100,000 sources in FP32, 24.9 ms (now 7.36 ms, matrix pipe 76 % and
 * vector unit 13 % busy; 7.96 ms with LDS addresses formed per k-step)
 * and, for 197 stations x 30,011 sources in FP64, 1.77 ms (now 0.85 ms,
 * 71 % and 10 %).
 *
 * The source range is split over workgroups; partial sums go to an FP64
 * workspace in accumulator order (coalesced) and a second kernel adds the
 * splits in a fixed order and scatters them to vis.  A single split writes
 * vis itself.
 */
#include <hip/hip_runtime.h>
#include <math.h>

#include "private.h"
#include "workspace.h"
#include "xcorr_common.h"

using namespace oskar_amd;

namespace {

constexpr int NT = 256;
constexpr int ROWS = 64;             /* rows per workgroup side */
constexpr int BLK = 16;              /* rows of an MFMA operand */
constexpr int WAVE_VALUES = 2048;    /* FP64 accumulators of a wave */
/* One k-step of one side: 4 row blocks x 4 x 16 values, and padding. */
constexpr int KSTRIDE = 4 * 4 * BLK + 2;

typedef double d4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));

template <typename FP> struct Acc;
template <> struct Acc<double> { using type = d4v; };
template <> struct Acc<float> { using type = f4v; };

__device__ __forceinline__ d4v mfma(double a, double b, d4v c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4v mfma(float a, float b, f4v c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
/* c - a b as mfma_minus(minus(a), b, c): FP64 instructions negate an
 * operand themselves (the blgp field's low bit: the first). */
__device__ __forceinline__ double minus(double a) { return a; }
__device__ __forceinline__ d4v mfma_minus(double a, double b, d4v c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 1);
}
__device__ __forceinline__ float minus(float a) { return -a; }
__device__ __forceinline__ f4v mfma_minus(float a, float b, f4v c)
{
    return mfma(a, b, c);
}

/* Row of accumulator register v in lane group g = lane / 16 (the column is
 * lane % 16). */
template <typename FP> __device__ __forceinline__ int acc_row(int v, int g)
{
    return sizeof(FP) == 8 ? 4 * v + g : 4 * g + v;
}

template <typename FP, bool MATRIX> struct Geo
{
    static constexpr int NR = MATRIX ? 8 : 2;      /* reals per value */
    static constexpr int RPS = MATRIX ? 2 : 1;     /* rows per station */
    static constexpr int SPK = MATRIX ? 1 : 2;     /* sources per k-step */
    static constexpr int KT = sizeof(FP) == 8 ? 8 : 16; /* k-steps, stage */
    static constexpr int PAIRS = KT / 2;
    static constexpr int TILE = KT * SPK;          /* sources per stage */
    static constexpr int BST = ROWS / RPS;         /* stations, workgroup */
    static constexpr int WST = BST / 2;            /* stations, wave */
    static constexpr int EPT = ROWS * KT / NT;     /* entries per thread */
    static constexpr int RPE = NT / KT;            /* rows between entries */
    /* The four contraction steps of an entry (two complex numbers) and
     * those of its neighbour make a pair of k-steps: the real parts of all
     * four numbers, then the imaginary parts.  Steps of a k-step between
     * the two entries, and between the numbers of one, so that the threads
     * of one store (neighbouring rows of KT entries) meet different banks,
     * with the padding of KSTRIDE. */
    static constexpr int ENTRY = sizeof(FP) == 8 ? BLK : 2 * BLK;
    static constexpr int NUMBER = 3 * BLK - ENTRY;
    static constexpr int SIDE = KT * KSTRIDE;
    static_assert(RPE % BLK == 0, "entries of a thread: whole row blocks");
};

/* Jones values need only the alignment of their reals. */
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

/* Four consecutive reals. */
__device__ __forceinline__ void load4(const float* a, float* x)
{
    const f4u v = *(const f4u*) a;
    x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
}
__device__ __forceinline__ void load2(const float* a, float* x)
{
    const f2u v = *(const f2u*) a;
    x[0] = v.x; x[1] = v.y;
}
__device__ __forceinline__ void load2(const double* a, double* x)
{
    const d2u v = *(const d2u*) a;
    x[0] = v.x; x[1] = v.y;
}
__device__ __forceinline__ void load4(const double* a, double* x)
{
    load2(a, x);
    load2(a + 2, x + 2);
}

/* What one thread stages: entry e of a side is operand row
 * row0 + e RPE at k-step kt, its four contraction steps: one row of a
 * station's matrix, or a station's scalars of two sources.  Consecutive
 * threads take consecutive addresses of a station's run of sources. */
template <typename FP, bool MATRIX> struct Stager
{
    using G = Geo<FP, MATRIX>;
    const FP *jp[G::EPT], *jq[G::EPT];
    FP p[G::EPT][4], q[G::EPT][4];
    FP flux[MATRIX ? 4 : 2];
    int kt, row0, slot;
    bool in[G::SPK];             /* source within the range */

    __device__ __forceinline__ void init(const XcorrArgs<FP>& A, int p0,
            int q0, int tid)
    {
        const int i = tid % G::RPS;
        kt = (tid / G::RPS) % G::KT;
        row0 = (tid / (G::RPS * G::KT)) * G::RPS + i;
        slot = (kt & ~1) * KSTRIDE + (kt & 1) * G::ENTRY +
                (row0 / BLK) * (4 * BLK) + row0 % BLK;
#pragma unroll
        for (int e = 0; e < G::EPT; ++e)
        {
            /* Rows of stations past the last repeat it; they belong to no
             * baseline. */
            const int st = (row0 + e * G::RPE) / G::RPS;
            const int last = A.num_stations - 1;
            jp[e] = (const FP*) A.jones + (size_t) min(p0 + st, last) *
                    A.num_sources * G::NR + 4 * i;
            jq[e] = (const FP*) A.jones + (size_t) min(q0 + st, last) *
                    A.num_sources * G::NR + 4 * i;
        }
    }

    /* The flux of this thread's k-step in the stage that starts at s_tile
     * (sources past the end repeat the last one). */
    __device__ __forceinline__ void load_flux(const XcorrArgs<FP>& A,
            int s_tile, int s_end)
    {
        const int s = s_tile + kt * G::SPK;
        const int sa = min(s, s_end - 1);
        in[0] = s < s_end;
        flux[0] = A.I[sa];
        if constexpr (MATRIX)
        {
            flux[1] = A.Q[sa];
            flux[2] = A.U[sa];
            flux[3] = A.V[sa];
        }
        else
        {
            in[1] = s + 1 < s_end;
            flux[1] = A.I[min(s + 1, s_end - 1)];
        }
    }

    __device__ __forceinline__ void load_entry(int e, int s_tile, int s_end)
    {
        const int s = s_tile + kt * G::SPK;
        const size_t sa = (size_t) min(s, s_end - 1);
        if constexpr (MATRIX)
        {
            load4(jp[e] + sa * 8, p[e]);
            load4(jq[e] + sa * 8, q[e]);
        }
        else
        {
            const size_t sb = (size_t) min(s + 1, s_end - 1);
            load2(jp[e] + 2 * sa, p[e]);
            load2(jp[e] + 2 * sb, p[e] + 2);
            load2(jq[e] + 2 * sa, q[e]);
            load2(jq[e] + 2 * sb, q[e] + 2);
        }
    }

    /* Forms an entry's M on the first side and writes both sides.  EDGE:
     * the stage may reach past the end, and the sources there are stored
     * as zeros. */
    template <bool EDGE>
    __device__ __forceinline__ void store_entry(int e, FP* side_p,
            FP* side_q) const
    {
        FP M[4];
        if constexpr (MATRIX)
            row_times_brightness<FP>(p[e], flux[0], flux[1], flux[2],
                    flux[3], M);
        else
        {
#pragma unroll
            for (int k = 0; k < 4; ++k) M[k] = p[e][k] * flux[k / 2];
        }
        const int o = slot + e * (G::RPE / BLK) * (4 * BLK);
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            const bool use = !EDGE || in[MATRIX ? 0 : k / 2];
            const int at = o + (k & 1) * KSTRIDE + (k >> 1) * G::NUMBER;
            side_p[at] = use ? M[k] : (FP) 0;
            side_q[at] = use ? q[e][k] : (FP) 0;
        }
    }

    __device__ __forceinline__ void load_all(const XcorrArgs<FP>& A,
            int s_tile, int s_end)
    {
        load_flux(A, s_tile, s_end);
#pragma unroll
        for (int e = 0; e < G::EPT; ++e) load_entry(e, s_tile, s_end);
    }

    __device__ __forceinline__ void store_all(FP* buf) const
    {
#pragma unroll
        for (int e = 0; e < G::EPT; ++e)
            store_entry<true>(e, buf, buf + G::SIDE);
    }
};

__device__ __forceinline__ int opaque(int x)
{
    asm volatile("" : "+v"(x));
    return x;
}

/* Operands of a pair of k-steps in a wave: real (0) and imaginary (1) parts
 * of its two row blocks on each side. */
template <typename FP> struct Operands
{
    FP x[2][2], w[2][2];

    /* LDS elements.  Volatile: the reads stay single ones, whose 16-bit
     * offsets hold the k-step (paired reads reach only 256 elements, and
     * need an address of their own per k-step). */
    typedef const volatile __attribute__((address_space(3))) FP* Lds;

    /* xp, wp: this lane's element of the wave's first blocks. */
    __device__ __forceinline__ void read(Lds xp, Lds wp)
    {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 2; ++r)
            {
                x[c][r] = xp[c * KSTRIDE + r * (4 * BLK)];
                w[c][r] = wp[c * KSTRIDE + r * (4 * BLK)];
            }
    }
};

/* A wave's FP accumulators of Re and Im. */
template <typename FP> struct Sums
{
    typedef typename Acc<FP>::type A;
    A re[2][2], im[2][2];

    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                re[b / 2][b % 2][v] = im[b / 2][b % 2][v] = (FP) 0;
    }

    /* Re += x_re w_re + x_im w_im, Im += x_im w_re - x_re w_im.
     * skip (wave-uniform): block (0, 1) holds no baseline.  FIRST: the sums
     * start here. */
    template <bool FIRST>
    __device__ __forceinline__ void multiply(const Operands<FP>& o,
            bool skip)
    {
        const A z = {(FP) 0, (FP) 0, (FP) 0, (FP) 0};
        const FP n[2] = {minus(o.x[0][0]), minus(o.x[0][1])};
#pragma unroll
        for (int b = 0; b < 3; ++b)
        {
            const int r = b > 0, c = b > 1;    /* (0,0), (1,0), (1,1) */
            re[r][c] = mfma(o.x[0][r], o.w[0][c], FIRST ? z : re[r][c]);
            im[r][c] = mfma(o.x[1][r], o.w[0][c], FIRST ? z : im[r][c]);
        }
        if (!skip)
        {
            re[0][1] = mfma(o.x[0][0], o.w[0][1], FIRST ? z : re[0][1]);
            im[0][1] = mfma(o.x[1][0], o.w[0][1], FIRST ? z : im[0][1]);
        }
#pragma unroll
        for (int b = 0; b < 3; ++b)
        {
            const int r = b > 0, c = b > 1;
            re[r][c] = mfma(o.x[1][r], o.w[1][c], re[r][c]);
            im[r][c] = mfma_minus(n[r], o.w[1][c], im[r][c]);
        }
        if (!skip)
        {
            re[0][1] = mfma(o.x[1][0], o.w[1][1], re[0][1]);
            im[0][1] = mfma_minus(n[0], o.w[1][1], im[0][1]);
        }
    }
};

/* FP64 sums over stages of the accumulators (FP32: each stage; FP64: up
 * to four stages, so that rounding grows with the square root of
 * the stages rather than of all products). */
template <typename FP> struct Totals
{
    double re[2][2][4], im[2][2][4];

    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            re[i / 8][(i / 4) % 2][i % 4] = im[i / 8][(i / 4) % 2][i % 4] =
                    0.0;
    }

    /* Adds value i of 16 (Re and Im). */
    __device__ __forceinline__ void add(const Sums<FP>& s, int i)
    {
        const int a = i / 8, b = (i / 4) % 2, v = i % 4;
        re[a][b][v] += (double) s.re[a][b][v];
        im[a][b][v] += (double) s.im[a][b][v];
    }
};

/* One stage of a workgroup whose four waves all have a full tile: the
 * products of buffer cur, the staging of the next buffer, the loads of the
 * stage after it and (FP32) the previous stage's additions to the FP64
 * totals, spread over the k-steps so that they issue between the MFMAs
 * (an MFMA occupies the matrix pipe for 8 or 16 issue slots of a wave). */
template <typename FP, bool MATRIX>
__device__ __forceinline__ void full_stage(const XcorrArgs<FP>& A,
        Stager<FP, MATRIX>& d, const FP* cur, FP* nxt, int s_after,
        int s_end, int lane, int wp, int wq, Sums<FP>& sums,
        const Sums<FP>& old, Totals<FP>& tot)
{
    using G = Geo<FP, MATRIX>;
    constexpr bool SINGLE = sizeof(FP) == 4;
    /* Opaque, so that the addresses of the k-steps are formed where they
     * are used instead of being held in registers across stages. */
    typedef typename Operands<FP>::Lds Lds;
    const Lds xp = (Lds) cur + opaque(wp * 2 * (4 * BLK) + lane);
    const Lds xq = (Lds) cur + opaque(G::SIDE + wq * 2 * (4 * BLK) + lane);
    constexpr int EVERY = G::PAIRS / G::EPT;
    static_assert(EVERY == 2, "an entry's store, then its next load");
    Operands<FP> o[2];
    o[0].read(xp, xq);
#pragma unroll
    for (int m = 0; m < G::PAIRS; ++m)
    {
        if (m + 1 < G::PAIRS)
            o[(m + 1) & 1].read(xp + 2 * (m + 1) * KSTRIDE,
                    xq + 2 * (m + 1) * KSTRIDE);
        if (m % EVERY == 0)
            d.template store_entry<false>(m / EVERY, nxt, nxt + G::SIDE);
        else
            d.load_entry(m / EVERY, s_after, s_end);
        if (m == G::PAIRS - 1) d.load_flux(A, s_after, s_end);
        if constexpr (SINGLE)
        {
            tot.add(old, 2 * m);
            tot.add(old, 2 * m + 1);
        }
        if (SINGLE && m == 0) sums.template multiply<true>(o[0], false);
        else sums.template multiply<false>(o[m & 1], false);
        __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, SINGLE ? 6 : 8, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

/* The products of one stage for pairs first, first + step, ... of k-steps. */
template <typename FP, bool MATRIX>
__device__ __forceinline__ void part_stage(const FP* cur, int lane, int wp,
        int wq, int first, int step, bool skip, Sums<FP>& sums)
{
    using G = Geo<FP, MATRIX>;
    const int at = first * 2 * KSTRIDE + lane;
    typedef typename Operands<FP>::Lds Lds;
    Lds xp = (Lds) cur + wp * 2 * (4 * BLK) + at;
    Lds xq = (Lds) cur + G::SIDE + wq * 2 * (4 * BLK) + at;
    const int inc = step * 2 * KSTRIDE;
    Operands<FP> o[2];
    o[0].read(xp, xq);
    /* Two pairs per iteration, each reading the next one's operands ahead
     * of its MFMAs (the last read repeats the last pair). */
    for (int m = first; m < G::PAIRS; m += 2 * step)
    {
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            if (m + h * step >= G::PAIRS) break;
            const int up = m + (h + 1) * step < G::PAIRS ? inc : 0;
            xp += up;
            xq += up;
            o[h ^ 1].read(xp, xq);
            __builtin_amdgcn_sched_barrier(0);
            sums.template multiply<false>(o[h], skip);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

/* Workgroup tiles (ib >= jb) of nb x nb station blocks. */
__host__ __device__ inline void tile_coords(int t, int* ib, int* jb)
{
    int i = 0;
    while (t > i) { t -= i + 1; ++i; }
    *ib = i;
    *jb = t;
}

/* What the four waves of a workgroup tile do.  A sub-tile (wp, wq) of
 * WST x WST stations is live if it holds a p > q pair of real stations.
 * With fewer than four live sub-tiles, and partial sums (shared), the
 * waves share them: wave w takes sub-tile w % live and every share-th
 * k-step of a stage, and the reduction adds the waves of a sub-tile. */
struct Roles
{
    int live, wp, wq, first, step;
    bool active;
};

__host__ __device__ inline Roles wave_roles(int N, int p0, int q0, int wst,
        int wave, bool shared)
{
    /* (1, 0) first: on a diagonal tile it is the one without a skipped
     * block, and of three sub-tiles the first gets two waves. */
    const int order[4] = {1, 0, 3, 2};          /* wp + 2 wq */
    int list[4] = {0, 0, 0, 0}, n = 0;
    for (int i = 0; i < 4; ++i)
    {
        const int wp = order[i] & 1, wq = order[i] >> 1;
        const int pl = (p0 + wp * wst + wst < N ? p0 + wp * wst + wst : N) -
                1;
        if (p0 + wp * wst < N && pl > q0 + wq * wst) list[n++] = order[i];
    }
    Roles r;
    r.live = n;
    const int u = n ? wave % n : 0;
    r.wp = list[u] & 1;
    r.wq = list[u] >> 1;
    r.step = shared && n ? (4 - u + n - 1) / n : 1;
    r.first = shared && n ? wave / n : 0;
    r.active = n > 0 && (shared || wave < n);
    return r;
}

/* The station pair and element (i, k) of accumulator register v of block
 * (rf, cf) in this lane; false if it is no p > q baseline. */
template <typename FP, bool MATRIX>
__device__ __forceinline__ bool acc_place(int N, int p0, int q0, int rf,
        int cf, int v, int lane, int* p, int* q, int* i, int* k)
{
    using G = Geo<FP, MATRIX>;
    const int row = rf * BLK + acc_row<FP>(v, lane >> 4);
    const int col = cf * BLK + (lane & 15);
    *p = p0 + row / G::RPS;
    *q = q0 + col / G::RPS;
    *i = row % G::RPS;
    *k = col % G::RPS;
    return *p < N && *p > *q;
}

/* The two reals of vis that element (i, k) of baseline (p, q) adds to, or
 * NULL outside the uv filter. */
template <typename FP, bool MATRIX>
__device__ __forceinline__ FP* vis_place(const XcorrArgs<FP>& A, int p, int q,
        int i, int k)
{
    using G = Geo<FP, MATRIX>;
    BaselineTerms<FP, false> t;
    t.init(A, p, q);
    if (t.uv_len < A.uv_min || t.uv_len > A.uv_max) return nullptr;
    /* CASA: element [i][k] = conj(V[k][i]). */
    const int el = MATRIX ? (A.use_casa ? 2 * k + i : 2 * i + k) : 0;
    return (FP*) A.vis + ((size_t) A.offset_out +
            baseline_index(A.num_stations, p, q)) * G::NR + 2 * el;
}

template <typename FP, bool MATRIX>
__global__ __launch_bounds__(NT, 2)
void xcorr_product_kernel(XcorrArgs<FP> A, int tiles)
{
    using G = Geo<FP, MATRIX>;
    __shared__ __align__(16) FP lds[2][2 * G::SIDE];
    /* Workgroup w runs on XCD w % 8; each XCD takes a contiguous range of
     * (split, tile) items, so the tiles of a split, which read the same
     * Jones values, share that XCD's L2.  A bijection for any grid. */
    const int total = (int) gridDim.x, w = (int) blockIdx.x;
    const int xq = total / 8, xr = total % 8, xcd = w % 8;
    const int item = xcd * xq + min(xcd, xr) + w / 8;
    const int tile = item % tiles, split = item / tiles;
    int ib, jb;
    tile_coords(tile, &ib, &jb);
    const int N = A.num_stations;
    const int p0 = ib * G::BST, q0 = jb * G::BST;
    const int s_begin = split * A.src_per_split;
    const int s_end = min(A.num_sources, s_begin + A.src_per_split);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Roles role = wave_roles(N, p0, q0, G::WST, wave,
            A.num_splits > 1);
    if (role.live == 0) return;
    const int wp = role.wp, wq = role.wq;
    const int wp0 = p0 + wp * G::WST, wq0 = q0 + wq * G::WST;

    constexpr bool SINGLE = sizeof(FP) == 4;
    Sums<FP> sums;
    Totals<FP> tot;
    sums.clear();
    tot.clear();
    Stager<FP, MATRIX> d;
    d.init(A, p0, q0, tid);
    d.load_all(A, s_begin, s_end);
    d.store_all(lds[0]);
    d.load_all(A, s_begin + G::TILE, s_end);
    __syncthreads();
    int s = s_begin;
    if (role.live == 4 && ib != jb)
    {
        /* Pairs of stages (each LDS buffer, and in FP32 each of two
         * accumulator sets, fixed in its copy of the body) while what they
         * stage is whole: the rest is left to the loop below. */
        Sums<FP> other;
        other.clear();
        for (int pair = 0; s + 3 * G::TILE <= s_end; s += 2 * G::TILE)
        {
            full_stage<FP, MATRIX>(A, d, lds[0], lds[1], s + 2 * G::TILE,
                    s_end, lane, wp, wq, sums, other, tot);
            __syncthreads();
            full_stage<FP, MATRIX>(A, d, lds[1], lds[0], s + 3 * G::TILE,
                    s_end, lane, wp, wq, SINGLE ? other : sums, sums, tot);
            if (!SINGLE && (++pair & 1) == 0)
            {
#pragma unroll
                for (int i = 0; i < 16; ++i) tot.add(sums, i);
                sums.clear();
            }
            __syncthreads();
        }
        if constexpr (SINGLE)
        {
#pragma unroll
            for (int i = 0; i < 16; ++i) tot.add(other, i);
            sums.clear();
        }
    }
    const bool skip = wp0 == wq0;
    for (int buf = 0; s < s_end; s += G::TILE)
    {
        if (role.active)
            part_stage<FP, MATRIX>(lds[buf], lane, wp, wq, role.first,
                    role.step, skip, sums);
#pragma unroll
        for (int i = 0; i < 16; ++i) tot.add(sums, i);
        sums.clear();
        /* The other buffer was last read before the last barrier. */
        buf ^= 1;
        if (s + G::TILE < s_end)
        {
            d.store_all(lds[buf]);
            d.load_all(A, s + 2 * G::TILE, s_end);
        }
        __syncthreads();
    }
    if (!role.active) return;
    if (A.num_splits > 1)
    {
        double* part = A.partial +
                (((size_t) split * tiles + tile) * 4 + wave) * WAVE_VALUES +
                lane;
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
            const int r = i / 8, c = (i / 4) % 2, v = i % 4;
            part[(i * 2 + 0) * 64] = tot.re[r][c][v];
            part[(i * 2 + 1) * 64] = tot.im[r][c][v];
        }
        return;
    }
    /* One split: vis itself, eight values at a time, all loaded before the
     * first is stored (a load and a store at a time are one chain: 3000
     * stations x 16 sources of FP64 matrices 290 -> 255 us, 512 x 60 38.2 ->
     * 36.6).  Through the LDS to consecutive accesses it was 10 % slower:
     * every lane then has the terms of twice as many baselines to form. */
#pragma unroll
    for (int h = 0; h < 2; ++h)
    {
        FP* at[8];
        FP old[8][2];
#pragma unroll
        for (int j = 0; j < 8; ++j)
        {
            int p, q, ei, ek;
            at[j] = acc_place<FP, MATRIX>(N, wp0, wq0, h, j / 4, j % 4,
                    lane, &p, &q, &ei, &ek) ?
                    vis_place<FP, MATRIX>(A, p, q, ei, ek) : nullptr;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (at[j])
            {
                old[j][0] = at[j][0];
                old[j][1] = at[j][1];
            }
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (at[j])
            {
                const double im = tot.im[h][j / 4][j % 4];
                at[j][0] = old[j][0] + (FP) tot.re[h][j / 4][j % 4];
                at[j][1] = old[j][1] + (FP) (A.use_casa ? -im : im);
            }
    }
}

/* Adds the splits in a fixed order and scatters the sums to vis.
 * Workgroup (x, y): accumulator register x = (rf, cf, v) of sub-tile y; its
 * GROUPS waves add a share of the splits each (consecutive lanes on
 * consecutive partials; the partials of all waves that share the sub-tile),
 * the shares are then added in order.  4 waves; 16 where there are few
 * sub-tiles, whose many splits (hundreds, of up to four waves each) would be
 * long chains on a chip that is idle (64 stations x 2,000 FP64 scalars 20 ->
 * 18 us, 30 x 2,000 matrices 23 -> 21). */
template <typename FP, bool MATRIX, int GROUPS>
__global__ __launch_bounds__(64 * GROUPS)
void xcorr_product_reduce_kernel(XcorrArgs<FP> A, int tiles)
{
    using G = Geo<FP, MATRIX>;
    __shared__ double sums[GROUPS - 1][2][64];
    const int N = A.num_stations;
    const int tile = blockIdx.y / 4, u = blockIdx.y % 4;
    int ib, jb;
    tile_coords(tile, &ib, &jb);
    const Roles role = wave_roles(N, ib * G::BST, jb * G::BST, G::WST, u,
            true);
    if (u >= role.live) return;
    const int reg = blockIdx.x;                 /* (rf * 2 + cf) * 4 + v */
    const int lane = threadIdx.x & 63, group = threadIdx.x >> 6;
    const size_t stride = (size_t) tiles * 4 * WAVE_VALUES;
    const double* part = A.partial + ((size_t) tile * 4 + u) * WAVE_VALUES +
            (size_t) reg * 128 + lane;
    const int per = (A.num_splits + GROUPS - 1) / GROUPS;
    const int k1 = min(A.num_splits, (group + 1) * per);
    double re = 0.0, im = 0.0;
    for (int h = 0; h < role.step; ++h)
    {
#pragma unroll 8
        for (int s = group * per; s < k1; ++s)
        {
            re += part[s * stride];
            im += part[s * stride + 64];
        }
        part += (size_t) role.live * WAVE_VALUES;
    }
    if (group > 0)
    {
        sums[group - 1][0][lane] = re;
        sums[group - 1][1][lane] = im;
    }
    __syncthreads();
    if (group > 0) return;
    for (int h = 0; h < GROUPS - 1; ++h)
    {
        re += sums[h][0][lane];
        im += sums[h][1][lane];
    }
    int p, q, i, k;
    if (acc_place<FP, MATRIX>(N, ib * G::BST + role.wp * G::WST,
            jb * G::BST + role.wq * G::WST, reg >> 3, (reg >> 2) & 1,
            reg & 3, lane, &p, &q, &i, &k))
    {
        FP* o = vis_place<FP, MATRIX>(A, p, q, i, k);
        if (!o) return;
        o[0] += (FP) re;
        o[1] += (FP) (A.use_casa ? -im : im);
    }
}

} /* namespace */

namespace oskar_amd {

template <typename FP, bool MATRIX>
hipError_t xcorr_product_launch(XcorrArgs<FP> A, hipStream_t stream,
        double* fixed)
{
    using G = Geo<FP, MATRIX>;
    if (A.num_stations < 2 || A.num_sources <= 0) return hipSuccess;
    const int nb = (A.num_stations + G::BST - 1) / G::BST;
    const int tiles = nb * (nb + 1) / 2;
    const int stages = (A.num_sources + G::TILE - 1) / G::TILE;
    /* Splits.  In units of the time a CU needs for one stage of one tile
     * (4096 matrix-core cycles, 1.75 us), k splits cost about stages / k for
     * the last workgroups to finish alone, and 0.026 k tiles for filling
     * each workgroup's pipeline (two stages on one of 256 CUs) and for its
     * 64 KB of partial sums written and read at 4 TB/s.  197 stations x 30011
     * sources in FP64: 71 splits against one round of 18. */
    const size_t split_bytes = (size_t) tiles * 4 * WAVE_VALUES *
            sizeof(double);
    const int most = max(1, (int) min((size_t) stages,
            XCORR_PARTIAL_BYTES / split_bytes));
    int splits = (int) sqrt(stages / (0.026 * tiles));
    splits = max(1, min(splits, most));
    const int per = (stages + splits - 1) / splits;
    splits = (stages + per - 1) / per;
    A.src_per_split = per * G::TILE;
    A.num_splits = splits;
    A.partial = nullptr;
    if (splits > 1)
    {
        A.partial = fixed;
        if (!fixed)
        {
            int dev = 0;
            hipError_t err = hipGetDevice(&dev);
            if (err != hipSuccess) return err;
            A.partial = (double*) ws_acquire(WS_XCORR_SPLIT, dev, stream,
                    (size_t) splits * split_bytes, &err);
            if (err != hipSuccess) return err;
        }
    }
    hipLaunchKernelGGL((xcorr_product_kernel<FP, MATRIX>),
            dim3((unsigned) (tiles * splits)), dim3(NT), 0, stream, A, tiles);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess || splits == 1) return err;
    const dim3 grid(16, (unsigned) (tiles * 4));
    if (tiles <= 3)
        hipLaunchKernelGGL((xcorr_product_reduce_kernel<FP, MATRIX, 16>),
                grid, dim3(64 * 16), 0, stream, A, tiles);
    else
        hipLaunchKernelGGL((xcorr_product_reduce_kernel<FP, MATRIX, 4>),
                grid, dim3(64 * 4), 0, stream, A, tiles);
    return hipGetLastError();
}

template hipError_t xcorr_product_launch<double, true>(XcorrArgs<double>,
        hipStream_t, double*);
template hipError_t xcorr_product_launch<double, false>(XcorrArgs<double>,
        hipStream_t, double*);
template hipError_t xcorr_product_launch<float, true>(XcorrArgs<float>,
        hipStream_t, double*);
template hipError_t xcorr_product_launch<float, false>(XcorrArgs<float>,
        hipStream_t, double*);

} /* namespace oskar_amd */
