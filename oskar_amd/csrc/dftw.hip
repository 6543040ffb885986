/*
 * Weighted DFT (array factor x element data) for gfx950.
 *
 * Computes, for each output direction j,
 *   out[j] = norm * sum_i data[idx_i][j] * w_i * exp(i k (x_j x_i + y_j y_i
 *            [+ z_j z_i]))
 * (oskar/math/define_dftw_c2c.h:24-77, define_dftw_m2m.h:24-107).
 *
 * Design:
 *  - One thread per output direction, 256 per workgroup.  Element weights,
 *    positions and data indices are staged through LDS in chunks of 256 and
 *    read as wavefront-uniform (broadcast) values.
 *  - The data index of element i is the same for every thread, so the sum
 *    is formed as a run-length product: consecutive elements that share a
 *    data index are summed into one complex array factor, which multiplies
 *    the (coalesced) data value once per run.  With one element type this
 *    reads the element pattern once per direction instead of once per
 *    element; with data_idx absent each element is its own run and the
 *    kernel reads data per element as the reference does.
 *  - Elements are staged with position and weight in one LDS record (a
 *    broadcast read per element).  A chunk whose elements all use one
 *    data row (the usual case: one element type, or long runs of one)
 *    skips the per-element run check and unrolls the element loop by 4.
 *  - Single precision carries the phase in revolutions (the wavenumber
 *    times 1/(2 pi) folded into the direction once per thread), reduces it
 *    to [-1/2, 1/2] and uses the hardware sine and cosine, which take
 *    revolutions; each term is four fused multiply-adds into the array
 *    factor.  Double precision reduces the phase to a quarter revolution and
 *    uses polynomials.
 */
#include <hip/hip_runtime.h>
#include <type_traits>

#include "device_common.h"
#include "dipole_device.h"
#include "private.h"

using namespace oskar_amd;

namespace {

constexpr int THREADS = 256;
constexpr int CHUNK = 256;

/* exp(i t) of the phase in the unit the kernel carries it in.  FP32 phases
 * are in revolutions for the hardware sine and cosine (which take
 * revolutions), reduced to [-1/2, 1/2] first unless DIRECT.  The hardware
 * reduces a phase of up to 256 revolutions exactly (the same errors against
 * the FP64 DFT with and without the reduction at up to 250 revolutions,
 * measured), so DIRECT serves when |t| is bounded below that: two fewer
 * instructions per term.  FP64 phases are in radians; DIRECT serves while
 * |t| is within the reduction of sincos_fold, past which its polynomials
 * leave their range without bound. */
template <bool DIRECT, typename FP>
__device__ __forceinline__ void phase_sincos(FP t, FP* s, FP* c)
{
    if constexpr (sizeof(FP) == 8)
    {
        sincos_fold(DIRECT ? t : far_phase(t), s, c);
    }
    else
    {
        const float r = DIRECT ? t : t - __builtin_rintf(t);
        *s = __builtin_amdgcn_sinf(r);
        *c = __builtin_amdgcn_cosf(r);
    }
}

/* Factor from k (x_out x_in + ...) to the kernel's phase unit. */
template <typename FP> constexpr double PHASE_UNIT =
        sizeof(FP) == 8 ? 1.0 : 0.15915494309189535;    /* 1 / (2 pi) */

/* One element of the chunk staged in LDS: position and weight. */
template <typename FP> struct Elem
{
    FP x, y, z, pad;
    Cplx<FP> w;
};

/* Largest |coordinate| of the chunk's elements, gathered in LDS as float
 * bits (non-negative floats order as unsigned integers); FP64: only whether
 * any is 2^25 or more (or no number), a store that no array makes. */
template <typename FP>
__device__ __forceinline__ void chunk_extent(unsigned int* bits, FP x, FP y,
        FP z)
{
    const FP a = fmax(fabs(x), fmax(fabs(y), fabs(z)));
    if constexpr (sizeof(FP) == 4) atomicMax(bits, __float_as_uint(a));
    else if (!(a < (FP) 0x1p25)) *bits = 1u;
}

/* Whether every phase of a thread's direction (xo, yo, zo, in phase units
 * per metre) over the chunk's elements takes phase_sincos's DIRECT form.
 * FP32: |t| <= (|xo| + |yo| + |zo|) ext + 1/2 (the weight's phase) < 255
 * revolutions; FP64: |t| < 2^50 radians. */
template <typename FP>
__device__ __forceinline__ bool direct_phase(FP xo, FP yo, FP zo,
        unsigned int bits)
{
    const FP sum = fabs(xo) + fabs(yo) + fabs(zo);
    if constexpr (sizeof(FP) == 4)
        return sum * __uint_as_float(bits) < 254.0f;
    else
        return sum < (FP) 0x1p25 && bits == 0u;
}

/* An element's weight in the form the terms use.  FP32: amplitude and
 * phase in revolutions, the phase then added into the element's phase by
 * the first fused multiply-add, so that a term takes two fused
 * multiply-adds into the array factor instead of the four of a complex
 * product (the weight's phase in FP32 revolutions errs by under 6e-8 of a
 * revolution, well under the FP32 phase of the element itself).  FP64:
 * the complex weight as it is. */
template <typename FP>
__device__ __forceinline__ Cplx<FP> term_weight(const Cplx<FP>& w)
{
    if constexpr (sizeof(FP) == 4)
    {
        Cplx<FP> p;
        p.x = sqrtf(w.x * w.x + w.y * w.y);
        p.y = atan2f(w.y, w.x) * 0.159154943091895336f;    /* 1 / (2 pi) */
        return p;
    }
    else
        return w;
}

/* Phase of a term: the direction (xo, yo, zo, already in phase units per
 * metre) dotted with the element's position, plus the FP32 weight's
 * phase. */
template <typename FP, bool IS_3D>
__device__ __forceinline__ FP term_phase(FP xo, FP yo, FP zo, FP ex, FP ey,
        FP ez, const Cplx<FP>& w)
{
    if constexpr (sizeof(FP) == 4)
    {
        float t = __builtin_fmaf(xo, ex, w.y);
        t = __builtin_fmaf(yo, ey, t);
        if (IS_3D) t = __builtin_fmaf(zo, ez, t);
        return t;
    }
    else
    {
        FP t = xo * ex + yo * ey;
        if (IS_3D) t += zo * ez;
        return t;
    }
}

/* af += w exp(i t), with w in term_weight's form and (s, c) the sine and
 * cosine of the term's phase. */
template <typename FP>
__device__ __forceinline__ void term_add(Cplx<FP>& af, const Cplx<FP>& w,
        FP s, FP c)
{
    if constexpr (sizeof(FP) == 4)
    {
        af.x = __builtin_fmaf(w.x, c, af.x);
        af.y = __builtin_fmaf(w.x, s, af.y);
    }
    else
    {
        af.x += w.x * c;
        af.x -= w.y * s;
        af.y += w.x * s;
        af.y += w.y * c;
    }
}

template <typename FP, bool MATRIX, bool IS_3D>
__global__ __launch_bounds__(THREADS)
void dftw_kernel(const int num_in, const FP wavenumber,
        const Cplx<FP>* __restrict__ weights, const FP* __restrict__ x_in,
        const FP* __restrict__ y_in, const FP* __restrict__ z_in,
        const int offset_coord_out, const int num_out,
        const FP* __restrict__ x_out, const FP* __restrict__ y_out,
        const FP* __restrict__ z_out, const int* __restrict__ data_idx,
        const Cplx<FP>* __restrict__ data, const int num_rows,
        const int eval_x, const int eval_y,
        const int offset_out, Cplx<FP>* __restrict__ output,
        const FP norm_factor)
{
    __shared__ Elem<FP> c_e[CHUNK];
    __shared__ int c_idx[CHUNK];
    __shared__ int c_uniform;
    __shared__ unsigned int c_ext;

    const int i_out = blockIdx.x * THREADS + threadIdx.x;
    const bool active = i_out < num_out;
    FP xo = (FP) 0, yo = (FP) 0, zo = (FP) 0;
    if (active)
    {
        const FP kk = wavenumber * (FP) PHASE_UNIT<FP>;
        xo = kk * x_out[i_out + offset_coord_out];
        yo = kk * y_out[i_out + offset_coord_out];
        if (IS_3D) zo = kk * z_out[i_out + offset_coord_out];
    }
    constexpr int NC = MATRIX ? 4 : 1;
    Cplx<FP> out[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) out[k].x = out[k].y = (FP) 0;
    Cplx<FP> af; af.x = af.y = (FP) 0;
    int run_idx = -1;

    /* Adds data[run_idx][i_out] * af to the outputs.  Indices outside the
     * num_rows rows held by data contribute nothing. */
    auto flush = [&]() {
        if (run_idx >= 0 && run_idx < num_rows && active)
        {
            const size_t base = (size_t) run_idx * num_out + i_out;
#pragma unroll
            for (int k = 0; k < NC; ++k)
            {
                if (MATRIX && ((k < 2 && !eval_x) || (k >= 2 && !eval_y)))
                    continue;
                const Cplx<FP> d = data[base * NC + k];
                out[k].x += d.x * af.x - d.y * af.y;
                out[k].y += d.y * af.x + d.x * af.y;
            }
        }
        af.x = af.y = (FP) 0;
    };
    /* af += w exp(i t) for element e. */
    auto term = [&](const Elem<FP>& e, auto direct) {
        const FP t = term_phase<FP, IS_3D>(xo, yo, zo, e.x, e.y, e.z, e.w);
        FP s, c;
        phase_sincos<decltype(direct)::value, FP>(t, &s, &c);
        term_add<FP>(af, e.w, s, c);
    };
    const std::true_type direct_t;
    const std::false_type reduce_t;

    for (int j = 0; j < num_in; j += CHUNK)
    {
        const int chunk = min(CHUNK, num_in - j);
        __syncthreads();
        if (threadIdx.x == 0)
        {
            c_uniform = 1;
            c_ext = 0u;
        }
        __syncthreads();
        for (int t = threadIdx.x; t < chunk; t += THREADS)
        {
            const int g = j + t;
            Elem<FP> e;
            e.x = x_in[g];
            e.y = y_in[g];
            e.z = IS_3D ? z_in[g] : (FP) 0;
            e.pad = (FP) 0;
            e.w = term_weight<FP>(weights[g]);
            c_e[t] = e;
            chunk_extent<FP>(&c_ext, e.x, e.y, e.z);
            const int idx = data_idx ? data_idx[g] : g;
            c_idx[t] = idx;
            /* Any element whose data row differs from the chunk's first
             * clears the flag (every writer stores the same value). */
            if (idx != (data_idx ? data_idx[j] : j)) c_uniform = 0;
        }
        __syncthreads();
        const bool direct = direct_phase<FP>(xo, yo, zo, c_ext);
        if (c_uniform)
        {
            /* One data row for the whole chunk: no run checks, and the
             * element loop unrolled. */
            const int idx = c_idx[0];
            if (idx != run_idx)
            {
                flush();
                run_idx = idx;
            }
            int i = 0;
            if (direct)
            {
                for (; i + 4 <= chunk; i += 4)
                {
#pragma unroll
                    for (int u = 0; u < 4; ++u) term(c_e[i + u], direct_t);
                }
                for (; i < chunk; ++i) term(c_e[i], direct_t);
            }
            else
            {
                for (; i + 4 <= chunk; i += 4)
                {
#pragma unroll
                    for (int u = 0; u < 4; ++u) term(c_e[i + u], reduce_t);
                }
                for (; i < chunk; ++i) term(c_e[i], reduce_t);
            }
        }
        else
        {
            for (int i = 0; i < chunk; ++i)
            {
                const int idx = c_idx[i];
                if (idx != run_idx)
                {
                    flush();
                    run_idx = idx;
                }
                if (direct) term(c_e[i], direct_t);
                else term(c_e[i], reduce_t);
            }
        }
    }
    flush();
    if (active)
    {
        const size_t o = (size_t) (i_out + offset_out) * NC;
#pragma unroll
        for (int k = 0; k < NC; ++k)
        {
            if (MATRIX && ((k < 2 && !eval_x) || (k >= 2 && !eval_y)))
                continue;
            Cplx<FP> v;
            v.x = out[k].x * norm_factor;
            v.y = out[k].y * norm_factor;
            output[o + k] = v;
        }
    }
}

/* An element of an aperture-array beam in LDS: position, and the weight in
 * term_weight's form. */
template <typename FP, bool IS_3D> struct AaElem;
template <typename FP> struct alignas(4 * sizeof(FP)) AaElem<FP, false>
{
    FP x, y;
    Cplx<FP> w;
    __device__ __forceinline__ FP at(FP xo, FP yo, FP) const
    {
        return term_phase<FP, false>(xo, yo, (FP) 0, x, y, (FP) 0, w);
    }
};
template <typename FP> struct alignas(4 * sizeof(FP)) AaElem<FP, true>
{
    FP x, y;
    Cplx<FP> w;
    FP z, pad[3];
    __device__ __forceinline__ FP at(FP xo, FP yo, FP zo) const
    {
        return term_phase<FP, true>(xo, yo, zo, x, y, z, w);
    }
};

struct AaGroup { oskar_AaStation st[OSKAR_AA_GROUP]; };

/* Beams of flat aperture-array stations whose elements are all of one
 * dipole type with a common orientation, in one pass per direction:
 * blockIdx.y = station of the group, D directions per thread (an element
 * read from LDS serves them all).  The array factor (dftw_kernel's sum, in
 * its order), times the direction's dipole pattern, times norm_factor, zero
 * below the horizon (blank_kernel's rule).  DFT weights without errors are
 * formed here, in FP64, from the measured positions and the pointing, once
 * per workgroup; others are read.  With NORM the result is divided as
 * oskar_mem_normalise divides by the beam in the normalisation direction,
 * whose pattern the host gives (norm_power) and whose array factor every
 * workgroup forms itself, each thread a stride of the elements, added in a
 * fixed order, so every workgroup of a station gets the same value.
 *
 * Bound: vector instructions: 4 and a hardware sine and cosine (FP32) or
 * 32 (FP64) per element and direction, and about 150 per direction for the
 * pattern and the output.  60 stations of 96 dipoles x 16,385 directions in
 * FP64: 1.8 ms as 60 launches of 65 workgroups with library sincos and
 * angles, 0.14 ms as 4 launches.  One station of 256 dipoles x 1M
 * directions in FP32: 78.3 -> 68.9 us (vector unit and transcendentals 80 %
 * of the time). */
template <typename FP, bool MATRIX, bool IS_3D, bool NORM, int D>
__global__ __launch_bounds__(THREADS)
void aa_beam_kernel(AaGroup G, const double wavenumber, const int num_out,
        const FP* __restrict__ x_out, const FP* __restrict__ y_out,
        const FP* __restrict__ z_out, Cplx<FP>* __restrict__ output)
{
    constexpr int NC = MATRIX ? 4 : 1;
    using E = AaElem<FP, IS_3D>;
    __shared__ E c_e[CHUNK];
    __shared__ FP red[2][THREADS / 64];
    __shared__ unsigned int c_ext;
    static_assert(D == 1 || D == 2, "directions per thread");
    const oskar_AaStation& S = G.st[blockIdx.y];
    const int tid = (int) threadIdx.x;
    const int num_in = S.num_elements;
    const double unit = wavenumber * PHASE_UNIT<FP>;
    const FP kk = (FP) unit;

    auto element = [&](int g) {
        E e;
        e.x = ((const FP*) S.x)[g];
        e.y = ((const FP*) S.y)[g];
        if constexpr (IS_3D) e.z = ((const FP*) S.z)[g];
        if (S.weights)
            e.w = term_weight<FP>(((const Cplx<FP>*) S.weights)[g]);
        else
        {
            double p = (double) ((const FP*) S.mx)[g] * S.beam_x +
                    (double) ((const FP*) S.my)[g] * S.beam_y +
                    (double) ((const FP*) S.mz)[g] * S.beam_z;
            if (S.cable) p += (double) ((const FP*) S.cable)[g];
            p *= -unit;
            if constexpr (sizeof(FP) == 4)
            {
                /* Whole revolutions taken off before the rounding. */
                e.w.x = 1.0f;
                e.w.y = (float) (p - rint(p));
            }
            else
                sincos_fold(far_phase(p), &e.w.y, &e.w.x);
        }
        return e;
    };

    FP scal = (FP) 1;
    if constexpr (NORM)
    {
        const FP xn = kk * (FP) S.nx, yn = kk * (FP) S.ny;
        const FP zn = kk * (FP) S.nz;
        Cplx<FP> a;
        a.x = a.y = (FP) 0;
        for (int g = tid; g < num_in; g += THREADS)
        {
            const E e = element(g);
            FP s, c;
            phase_sincos<false, FP>(e.at(xn, yn, zn), &s, &c);
            term_add<FP>(a, e.w, s, c);
        }
        FP re = a.x, im = a.y;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
        {
            re += __shfl_xor(re, o);
            im += __shfl_xor(im, o);
        }
        if ((tid & 63) == 0)
        {
            red[0][tid >> 6] = re;
            red[1][tid >> 6] = im;
        }
        __syncthreads();
        re = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
        im = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
        const FP f = (FP) S.norm_factor;
        const FP amp = (re * re + im * im) * (f * f) * (FP) S.norm_power;
        scal = (FP) 1 / sqrt(amp);
    }

    FP xo[D], yo[D], zo[D];
    Cplx<FP> af[D];
    const int first = (int) blockIdx.x * (THREADS * D) + tid;
#pragma unroll
    for (int d = 0; d < D; ++d)
    {
        const int i = min(first + d * THREADS, num_out - 1);
        xo[d] = kk * x_out[i];
        yo[d] = kk * y_out[i];
        zo[d] = IS_3D ? kk * z_out[i] : (FP) 0;
        af[d].x = af[d].y = (FP) 0;
    }
    /* Directions d0 .. d1 - 1 of the thread over the staged elements. */
    auto sum = [&](int chunk, auto direct, auto d0, auto d1) {
        auto term = [&](const E& e) {
#pragma unroll
            for (int d = decltype(d0)::value; d < decltype(d1)::value; ++d)
            {
                FP s, c;
                phase_sincos<decltype(direct)::value, FP>(
                        e.at(xo[d], yo[d], zo[d]), &s, &c);
                term_add<FP>(af[d], e.w, s, c);
            }
        };
        int i = 0;
        /* FP64's other form is for phases that no array reaches. */
        if (sizeof(FP) == 4 || decltype(direct)::value)
        {
            for (; i + 4 <= chunk; i += 4)
            {
#pragma unroll
                for (int u = 0; u < 4; ++u) term(c_e[i + u]);
            }
        }
#pragma unroll 1
        for (; i < chunk; ++i) term(c_e[i]);
    };
    const std::integral_constant<int, 0> d_0;
    const std::integral_constant<int, 1> d_1;
    const std::integral_constant<int, D> d_all;
    for (int j = 0; j < num_in; j += CHUNK)
    {
        const int chunk = min(CHUNK, num_in - j);
        __syncthreads();
        if (tid == 0) c_ext = 0u;
        __syncthreads();
        for (int t = tid; t < chunk; t += THREADS)
        {
            const E e = element(j + t);
            c_e[t] = e;
            FP z = (FP) 0;
            if constexpr (IS_3D) z = e.z;
            chunk_extent<FP>(&c_ext, e.x, e.y, z);
        }
        __syncthreads();
        /* Whether a direction's phases need the reduction depends on that
         * direction only, so that its value does not depend on D (FP64 phases
         * in DIRECT's range have the same value in both forms). */
        bool direct[D];
#pragma unroll
        for (int d = 0; d < D; ++d)
            direct[d] = direct_phase<FP>(xo[d], yo[d], zo[d], c_ext);
        if (direct[0] && direct[D - 1])
            sum(chunk, std::true_type(), d_0, d_all);
        else if (sizeof(FP) == 8 || (!direct[0] && !direct[D - 1]))
            sum(chunk, std::false_type(), d_0, d_all);
        else if (direct[0])
        {
            sum(chunk, std::true_type(), d_0, d_1);
            sum(chunk, std::false_type(), d_1, d_all);
        }
        else
        {
            sum(chunk, std::false_type(), d_0, d_1);
            sum(chunk, std::true_type(), d_1, d_all);
        }
    }
    const DipoleParams<FP> P = {(FP) S.kL, (FP) S.cos_dx,
            (FP) S.sin_dx, (FP) S.cos_dy, (FP) S.sin_dy, S.swap_xy};
#pragma unroll
    for (int d = 0; d < D; ++d)
    {
        const int i = first + d * THREADS;
        if (i >= num_out) break;
        const FP z = z_out[i];
        Cplx<FP> e[NC];
        dipole_enu_point<FP, MATRIX>(x_out[i], y_out[i], z, P, e, 0);
        const FP f = (FP) S.norm_factor;
        Cplx<FP>* o = output + (S.offset + (size_t) i) * NC;
#pragma unroll
        for (int k = 0; k < NC; ++k)
        {
            Cplx<FP> v;
            v.x = z < (FP) 0 ? (FP) 0 : e[k].x * af[d].x * f;
            v.y = z < (FP) 0 ? (FP) 0 : e[k].x * af[d].y * f;
            if constexpr (NORM)
            {
                v.x *= scal;
                v.y *= scal;
            }
            o[k] = v;
        }
    }
}

template <typename FP, bool MATRIX, bool IS_3D, bool NORM>
hipError_t aa_beam_t(const AaGroup& G, int count, double wavenumber,
        int num_out, const void* x_out, const void* y_out,
        const void* z_out, void* output, hipStream_t stream)
{
    /* Two directions per thread where that still gives every CU four
     * workgroups (an element's LDS reads and the workgroup's weights and
     * normalisation serve both); one otherwise. */
    const long long pairs = ((long long) num_out + 2 * THREADS - 1) /
            (2 * THREADS);
#define AA_LAUNCH(D) hipLaunchKernelGGL( \
        (aa_beam_kernel<FP, MATRIX, IS_3D, NORM, D>), \
        dim3((num_out + THREADS * D - 1) / (THREADS * D), count), \
        dim3(THREADS), 0, stream, G, wavenumber, num_out, \
        (const FP*) x_out, (const FP*) y_out, (const FP*) z_out, \
        (Cplx<FP>*) output)
    if (pairs * count >= 4 * 256) AA_LAUNCH(2);
    else AA_LAUNCH(1);
#undef AA_LAUNCH
    return hipGetLastError();
}

template <typename FP>
hipError_t launch_fp(int matrix, int is_3d, int num_in, double wavenumber,
        const void* weights, const void* x_in, const void* y_in,
        const void* z_in, int offset_coord_out, int num_out,
        const void* x_out, const void* y_out, const void* z_out,
        const int* data_idx, const void* data, int num_rows, int eval_x,
        int eval_y, int offset_out, void* output, double norm_factor,
        hipStream_t stream)
{
    if (num_out <= 0) return hipSuccess;
    const dim3 grid((num_out + THREADS - 1) / THREADS);
#define DFTW_ARGS num_in, (FP) wavenumber, (const Cplx<FP>*) weights,       \
        (const FP*) x_in, (const FP*) y_in, (const FP*) z_in,               \
        offset_coord_out, num_out, (const FP*) x_out, (const FP*) y_out,    \
        (const FP*) z_out, data_idx, (const Cplx<FP>*) data, num_rows,      \
        eval_x, eval_y,                                                     \
        offset_out, (Cplx<FP>*) output, (FP) norm_factor
    if (matrix && is_3d)
        hipLaunchKernelGGL((dftw_kernel<FP, true, true>), grid, dim3(THREADS),
                0, stream, DFTW_ARGS);
    else if (matrix)
        hipLaunchKernelGGL((dftw_kernel<FP, true, false>), grid,
                dim3(THREADS), 0, stream, DFTW_ARGS);
    else if (is_3d)
        hipLaunchKernelGGL((dftw_kernel<FP, false, true>), grid,
                dim3(THREADS), 0, stream, DFTW_ARGS);
    else
        hipLaunchKernelGGL((dftw_kernel<FP, false, false>), grid,
                dim3(THREADS), 0, stream, DFTW_ARGS);
#undef DFTW_ARGS
    return hipGetLastError();
}

} /* namespace */

extern "C" int oskar_amd_dftw_launch(int precision, int matrix, int is_3d,
        int num_in, double wavenumber, const void* weights,
        const void* x_in, const void* y_in, const void* z_in,
        int offset_coord_out, int num_out, const void* x_out,
        const void* y_out, const void* z_out, const int* data_idx,
        const void* data, int num_rows, int eval_x, int eval_y,
        int offset_out, void* output, double norm_factor, void* stream)
{
    if (precision == OSKAR_DOUBLE)
        return (int) launch_fp<double>(matrix, is_3d, num_in, wavenumber,
                weights, x_in, y_in, z_in, offset_coord_out, num_out, x_out,
                y_out, z_out, data_idx, data, num_rows, eval_x, eval_y,
                offset_out, output, norm_factor, (hipStream_t) stream);
    return (int) launch_fp<float>(matrix, is_3d, num_in, wavenumber,
            weights, x_in, y_in, z_in, offset_coord_out, num_out, x_out,
            y_out, z_out, data_idx, data, num_rows, eval_x, eval_y,
            offset_out, output, norm_factor, (hipStream_t) stream);
}

extern "C" int oskar_amd_aa_beam_launch(int precision, int matrix,
        int is_3d, int normalise, const oskar_AaStation* stations, int count,
        double wavenumber, int num_out, const void* x_out,
        const void* y_out, const void* z_out, void* output, void* stream)
{
    if (num_out <= 0 || count <= 0) return 0;
    if (count > OSKAR_AA_GROUP) return (int) hipErrorInvalidValue;
    const hipStream_t s = (hipStream_t) stream;
    AaGroup G;
    for (int i = 0; i < count; ++i) G.st[i] = stations[i];
    for (int i = count; i < OSKAR_AA_GROUP; ++i) G.st[i] = stations[0];
#define AB(FP, M, D, N) return (int) aa_beam_t<FP, M, D, N>(G, count, \
        wavenumber, num_out, x_out, y_out, z_out, output, s)
#define AF(FP, M, D) { if (normalise) AB(FP, M, D, true); AB(FP, M, D, false); }
    if (precision == OSKAR_DOUBLE)
    {
        if (matrix) { if (is_3d) AF(double, true, true) AF(double, true, false) }
        if (is_3d) AF(double, false, true)
        AF(double, false, false)
    }
    if (matrix) { if (is_3d) AF(float, true, true) AF(float, true, false) }
    if (is_3d) AF(float, false, true)
    AF(float, false, false)
#undef AF
#undef AB
}
