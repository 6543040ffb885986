/*
 * Arguments and per-baseline terms shared by the direct correlator's
 * kernels: the per-baseline sums (xcorr_direct.hip) and the matrix-core
 * product for point sources without smearing (xcorr_product.hip).
 */
#ifndef OSKAR_AMD_XCORR_COMMON_H_
#define OSKAR_AMD_XCORR_COMMON_H_

#include <hip/hip_runtime.h>
#include <stddef.h>

#include "device_common.h"

namespace oskar_amd {

constexpr double OMEGA_EARTH = 7.272205217e-5; /* rad/s, define_correlate_utils.h:3 */

/* Most FP64 partial sums of a call, in the stream's workspace or in the fixed
 * array of the allocation-free entry point, which has room for as many, so
 * that it splits the sources, and rounds, as oskar_cross_correlate does.  At
 * 512 stations of matrices a split is 8.4 MB (8.9 MB in the product): 30 fit,
 * eight rounds of workgroups.  20,000 extended sources with smearing in FP32
 * take 5.1 ms, 5.3 with half as many splits and 6.1 with a quarter; 100,000
 * point sources 7.4, 7.4 and 8.0. */
constexpr size_t XCORR_PARTIAL_BYTES = (size_t) 256 << 20;

template <typename FP>
struct XcorrArgs
{
    int num_sources, num_stations, offset_out, use_casa;
    int src_per_split, num_splits;
    const void* jones;
    const FP *I, *Q, *U, *V, *l, *m, *n, *a, *b, *c;
    const FP *st_u, *st_v, *st_w, *st_x, *st_y;
    FP uv_min, uv_max, inv_wl, frac_bw, time_int;
    FP sin_ha, cos_ha, sin_dec, cos_dec;    /* of the phase centre */
    void* vis;
    double* partial;
};

/* Baseline-dependent terms, written exactly as OSKAR_BASELINE_TERMS and
 * OSKAR_BASELINE_DELTAS (define_correlate_utils.h:5-26) with p = SP, q = SQ. */
template <typename FP, bool TS>
struct BaselineTerms
{
    FP uu, vv, ww, uu2, vv2, uuvv, uv_len, du, dv, dw;

    __device__ __forceinline__ void init(const XcorrArgs<FP>& A, int sp,
            int sq)
    {
        uu = (A.st_u[sp] - A.st_u[sq]) * A.inv_wl;
        vv = (A.st_v[sp] - A.st_v[sq]) * A.inv_wl;
        ww = (A.st_w[sp] - A.st_w[sq]) * A.inv_wl;
        uu2 = uu * uu;
        vv2 = vv * vv;
        uv_len = sqrt(uu2 + vv2);
        uuvv = 2 * uu * vv;
        const FP f = pi_v<FP>() * A.frac_bw;
        uu *= f; vv *= f; ww *= f;
        du = dv = dw = (FP) 0;
        if (TS)
        {
            FP temp = pi_v<FP>() * A.inv_wl;
            const FP xx = (A.st_x[sp] - A.st_x[sq]) * temp;
            const FP yy = (A.st_y[sp] - A.st_y[sq]) * temp;
            const FP rot = ((FP) OMEGA_EARTH) * A.time_int;
            temp = (xx * A.sin_ha + yy * A.cos_ha) * rot;
            du = (xx * A.cos_ha - yy * A.sin_ha) * rot;
            dv = temp * A.sin_dec;
            dw = -temp * A.cos_dec;
        }
    }
};

/* A run of VR reals moved by one load or store. */
template <typename FP, int VR> struct alignas(VR * sizeof(FP)) Vec
{
    FP v[VR];
};

/* One row (j0, j1) of M = J B with B = [[I+Q, U+iV], [U-iV, I-Q]]
 * (define_correlate_utils.h:36-39, define_multiply.h:69-87); 4 reals. */
template <typename FP>
__device__ __forceinline__ void row_times_brightness(const FP* j, FP I,
        FP Q, FP U, FP V, FP* M)
{
    const FP ba = I + Q, bd = I - Q;
    /* j0*ba + j1*conj(U+iV) */
    M[0] = j[0] * ba + (j[2] * U + j[3] * V);
    M[1] = j[1] * ba + (j[3] * U - j[2] * V);
    /* j1*bd + j0*(U+iV) */
    M[2] = j[2] * bd + (j[0] * U - j[1] * V);
    M[3] = j[3] * bd + (j[0] * V + j[1] * U);
}

/* Index of baseline (p, q), p > q (define_correlate_utils.h:42-43). */
__device__ __forceinline__ int baseline_index(int N, int p, int q)
{
    return q * (N - 1) - (q - 1) * q / 2 + p - q - 1;
}

/* xcorr_scratch.hip: the current device's fixed array of
 * XCORR_PARTIAL_BYTES. */
hipError_t xcorr_scratch(double** out);

/* xcorr_product.hip: the launch of the matrix-core product.  fixed: the
 * allocation-free entry point's array of XCORR_PARTIAL_BYTES, or NULL for
 * the per-stream workspace. */
template <typename FP, bool MATRIX>
hipError_t xcorr_product_launch(XcorrArgs<FP> A, hipStream_t stream,
        double* fixed);

} /* namespace oskar_amd */

#endif /* OSKAR_AMD_XCORR_COMMON_H_ */
