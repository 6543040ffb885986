/*
 * Device-side helpers shared by the HIP kernels of this library (gfx950).
 * Complex and 2x2 complex-matrix value types with the memory layout of the
 * reference's float2/double2 and float4c/double4c
 * (oskar/utility/oskar_vector_types.h:85,98), plus the smearing functions.
 */
#ifndef OSKAR_AMD_DEVICE_COMMON_H_
#define OSKAR_AMD_DEVICE_COMMON_H_

#include <hip/hip_runtime.h>

namespace oskar_amd {

template <typename FP> struct Cplx { FP x, y; };
template <typename FP> struct Mat4 { Cplx<FP> a, b, c, d; };

/* pi in each precision; the reference uses ((FP) M_PI). */
template <typename FP> __device__ __forceinline__ FP pi_v();
template <> __device__ __forceinline__ float pi_v<float>()
{ return 3.14159265358979323846f; }
template <> __device__ __forceinline__ double pi_v<double>()
{ return 3.14159265358979323846; }

/*
 * sinc(x) = sin(x)/x with sinc(0) = 1
 * (oskar/utility/oskar_kernel_macros.h:281), in the forms of the
 * correlator's inner loop, chosen by the largest |x| of a wave:
 *   |x| <= SMALL  polynomial in x^2, exactly 1 at 0;
 *   |x| <= MID    polynomial in x^2 - 8 (centred, so that its terms stay
 *                 below 1);
 *   |x| <= WIDE   sin(r) / x with r = x - k pi (two-part pi, k from the low
 *                 bits of a sum) and sin(r) = r sinc(r), which is the result
 *                 itself for k = 0;
 *   otherwise     the same with r = x - k pi (two-part pi, reduced twice
 *                 so that a rounded k does no harm) in [-pi/2, pi/2] and
 *                 sin(r) = r sinc(r); zero past LARGE, where |sinc| is
 *                 below the precision's roundoff.
 * The polynomials interpolate sin(x)/x at Chebyshev nodes (formed in
 * extended precision).  Largest and RMS error over 4e5 random arguments, in
 * units of 1e-8 (FP32) and 1e-17 (FP64): small 7.9 and 2.0, 14 and 3.6; mid
 * 11 and 2.3, 21 and 4.3; wide 11 and 1.6, 20 and 3.1 over |x| <= 4 and less
 * beyond; a correctly rounded sin(x) / x has 8.8 and 2.7, 16 and 5.0.  They
 * take 5, 8 and 20 instructions (FP32), 9, 12 and 30 (FP64); a
 * library sine and division, taken beside a series for small x by the lanes
 * of a wave, took about 35 and 250.
 */
template <typename FP> struct Sinc;
__device__ __forceinline__ float quotient(float a, float b);
__device__ __forceinline__ double quotient(double a, double b);

template <> struct Sinc<float>
{
    static constexpr float SMALL = 1.6f, MID = 4.0f, WIDE = 1e5f;
    static constexpr float LARGE = 3e7f;

    static __device__ __forceinline__ float small(float x)
    {
        const float y = x * x;
        float p = 2.630318022e-6f;
        p = fmaf(p, y, -1.982134418e-4f);
        p = fmaf(p, y, 8.333231322e-3f);
        p = fmaf(p, y, -1.666666567e-1f);
        return fmaf(p, y, 1.0f);
    }
    static __device__ __forceinline__ float mid(float x)
    {
        const float y = fmaf(x, x, -8.0f);
        float p = -6.034402578e-13f;
        p = fmaf(p, y, 1.227582758e-10f);
        p = fmaf(p, y, -1.829498686e-8f);
        p = fmaf(p, y, 1.894872298e-6f);
        p = fmaf(p, y, -1.247228211e-4f);
        p = fmaf(p, y, 4.510723520e-3f);
        p = fmaf(p, y, -6.626768410e-2f);
        return fmaf(p, y, 1.089198068e-1f);
    }
    static __device__ __forceinline__ float wide(float x)
    {
        const float m = fmaf(x, 0.318309886f, 12582912.0f);   /* 1.5 2^23 */
        const float k = m - 12582912.0f;
        float r = fmaf(-k, 3.14159274f, x);
        r = fmaf(-k, -8.74227766e-8f, r);
        const float p = small(r);
        const float s = __uint_as_float(__float_as_uint(r * p) ^
                (__float_as_uint(m) << 31));
        return k == 0.0f ? p : quotient(s, x);
    }
    static __device__ __forceinline__ float large(float x)
    {
        float k = rintf(x * 0.318309886f);
        float r = fmaf(-k, 3.14159274f, x);
        r = fmaf(-k, -8.74227766e-8f, r);
        const float k2 = rintf(r * 0.318309886f);
        r = fmaf(-k2, 3.14159274f, r);
        r = fmaf(-k2, -8.74227766e-8f, r);
        k += k2;
        const float s = r * small(r);
        const float q = (k - 2.0f * floorf(0.5f * k) != 0.0f ? -s : s) / x;
        return fabsf(x) > LARGE ? 0.0f * x : k == 0.0f ? small(x) : q;
    }
};

template <> struct Sinc<double>
{
    static constexpr double SMALL = 1.6, MID = 4.0, WIDE = 1e10;
    static constexpr double LARGE = 1e15;

    static __device__ __forceinline__ double small(double x)
    {
        const double y = x * x;
        double p = 2.7293211799890133e-15;
        p = fma(p, y, -7.643812566137517e-13);
        p = fma(p, y, 1.6058973007043202e-10);
        p = fma(p, y, -2.505210756706781e-8);
        p = fma(p, y, 2.755731921900734e-6);
        p = fma(p, y, -1.9841269841256248e-4);
        p = fma(p, y, 8.333333333333325e-3);
        p = fma(p, y, -1.6666666666666666e-1);
        return fma(p, y, 1.0);
    }
    static __device__ __forceinline__ double mid(double x)
    {
        const double y = fma(x, x, -8.0);
        double p = -3.2945201003283024e-23;
        p = fma(p, y, 1.6438941896768578e-20);
        p = fma(p, y, -6.783958446847399e-18);
        p = fma(p, y, 2.272799916310523e-15);
        p = fma(p, y, -6.025715437037218e-13);
        p = fma(p, y, 1.2246716537142188e-10);
        p = fma(p, y, -1.8295021639263917e-08);
        p = fma(p, y, 1.8948839015865714e-06);
        p = fma(p, y, -0.0001247228270651316);
        p = fma(p, y, 0.004510723318526139);
        p = fma(p, y, -0.06626768357401747);
        return fma(p, y, 0.10891980905843206);
    }
    static __device__ __forceinline__ double wide(double x)
    {
        const double m = fma(x, 0.31830988618379067, 6755399441055744.0);
        const double k = m - 6755399441055744.0;
        double r = fma(-k, 3.141592653589793, x);
        r = fma(-k, 1.2246467991473532e-16, r);
        const double p = small(r), s = r * p;
        const double q = quotient(__hiloint2double(__double2hiint(s) ^
                (__double2loint(m) << 31), __double2loint(s)), x);
        return k == 0.0 ? p : q;
    }
    static __device__ __forceinline__ double large(double x)
    {
        double k = rint(x * 0.31830988618379067);
        double r = fma(-k, 3.141592653589793, x);
        r = fma(-k, 1.2246467991473532e-16, r);
        const double k2 = rint(r * 0.31830988618379067);
        r = fma(-k2, 3.141592653589793, r);
        r = fma(-k2, 1.2246467991473532e-16, r);
        k += k2;
        const double s = r * small(r);
        const double q = (k - 2.0 * floor(0.5 * k) != 0.0 ? -s : s) / x;
        return fabs(x) > LARGE ? 0.0 * x : k == 0.0 ? small(x) : q;
    }
};

/* sin and cos of x: r = x - k pi in [-pi/2, pi/2] (k from the low bits of a
 * sum with 1.5 2^52, two-part pi), polynomials in r^2 that interpolate
 * sin(r) / r and cos(r) at Chebyshev nodes (formed in extended precision),
 * both negated for odd k.  Largest and RMS error over 5e5 random r: 2.4e-16
 * and 4.4e-17 (sine), 1.8e-16 and 3.9e-17 (cosine); 26 instructions where
 * the library's sincos took about 100.  For |x| up to 2^50 (whose rounding
 * is an eighth of a radian); far_phase takes larger ones there. */
__device__ __forceinline__ void sincos_fold(double x, double* s, double* c)
{
    const double m = fma(x, 0.31830988618379067, 6755399441055744.0);
    const double k = m - 6755399441055744.0;
    double r = fma(-k, 3.141592653589793, x);
    r = fma(-k, 1.2246467991473532e-16, r);
    const int sign = __double2loint(m) << 31;
    const double y = r * r;
    double ps = 2.731901991295671e-15;
    ps = fma(ps, y, -7.644016021446303e-13);
    ps = fma(ps, y, 1.605897917453392e-10);
    ps = fma(ps, y, -2.505210765661666e-08);
    ps = fma(ps, y, 2.7557319219632427e-06);
    ps = fma(ps, y, -0.00019841269841258002);
    ps = fma(ps, y, 0.008333333333333325);
    ps = fma(ps, y, -0.16666666666666666);
    ps = fma(ps, y, 1.0);
    double pc = 4.627703831606997e-14;
    pc = fma(pc, y, -1.146469250716007e-11);
    pc = fma(pc, y, 2.0876630965308777e-09);
    pc = fma(pc, y, -2.7557317769149775e-07);
    pc = fma(pc, y, 2.4801587292463866e-05);
    pc = fma(pc, y, -0.0013888888888860791);
    pc = fma(pc, y, 0.04166666666666634);
    pc = fma(pc, y, -0.5);
    pc = fma(pc, y, 1.0);
    ps *= r;
    *s = __hiloint2double(__double2hiint(ps) ^ sign, __double2loint(ps));
    *c = __hiloint2double(__double2hiint(pc) ^ sign, __double2loint(pc));
}

/* x less whole revolutions, for sincos_fold: within 2^-105 |x| of the angle
 * for |x| up to 2^100, 0 beyond (where the library's sincos reduces with as
 * many bits of pi as it takes, in registers that the beam's kernels need: 96
 * -> 177 with it).  An infinite x gives no number. */
__device__ __forceinline__ double far_phase(double x)
{
    if (fabs(x) < 0x1p50) return x;
    const double k = rint(x * 0.15915494309189535);
    double r = fma(-k, 6.283185307179586, x);
    r = fma(-k, 2.4492935982947064e-16, r);
    return fabs(r) < 0x1p50 ? r : 0.0 * r;
}

/* sin(x): r = x - k pi in [-pi/2, pi/2] (k from the low bits of a sum with
 * 1.5 2^23 in FP32, two-part pi), r sinc(r) negated for odd k.  FP32:
 * relative error below 1.5e-7 for |x| up to 2 pi (4.4e-7 up to 32, next to
 * the multiples of pi too), absolute below 1.7e-7 up to 1e6, against all
 * floats next to the multiples and 4e6 random ones; a reduction in rounded
 * revolutions erred by 1.0 of the value next to 2 pi and by 2.8e-6 at 32.
 * FP64: sincos_fold's sine. */
__device__ __forceinline__ double sin_fold(double x)
{
    double s, c;
    sincos_fold(x, &s, &c);
    return s;
}
__device__ __forceinline__ float sin_fold(float x)
{
    const float m = fmaf(x, 0.318309886f, 12582912.0f);
    const float k = m - 12582912.0f;
    float r = fmaf(-k, 3.14159274f, x);
    r = fmaf(-k, -8.74227766e-8f, r);
    return __uint_as_float(__float_as_uint(r * Sinc<float>::small(r)) ^
            (__float_as_uint(m) << 31));
}

/* 1 / sqrt(x) for normal x: the hardware estimate (1 ulp in FP32, about
 * 2^-26 in FP64) and Newton steps. */
__device__ __forceinline__ float inv_sqrt(float x)
{
    const float y = __builtin_amdgcn_rsqf(x);
    return fmaf(0.5f * y, fmaf(-x * y, y, 1.0f), y);
}
__device__ __forceinline__ double inv_sqrt(double x)
{
    double y = __builtin_amdgcn_rsq(x);
    y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
    return fma(0.5 * y, fma(-x * y, y, 1.0), y);
}

/* a / b for a normal b: the reciprocal's estimate and a Newton step (two in
 * FP64), then the quotient's remainder. */
__device__ __forceinline__ float quotient(float a, float b)
{
    float r = __builtin_amdgcn_rcpf(b);
    r = fmaf(fmaf(-b, r, 1.0f), r, r);
    const float q = a * r;
    return fmaf(fmaf(-b, q, a), r, q);
}
__device__ __forceinline__ double quotient(double a, double b)
{
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.0), r, r);
    r = fma(fma(-b, r, 1.0), r, r);
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

template <typename FP> __device__ __forceinline__ void sincos_v(FP x,
        FP* s, FP* c);
template <> __device__ __forceinline__ void sincos_v<float>(float x,
        float* s, float* c) { sincosf(x, s, c); }
template <> __device__ __forceinline__ void sincos_v<double>(double x,
        double* s, double* c) { sincos(x, s, c); }

} /* namespace oskar_amd */

#endif /* OSKAR_AMD_DEVICE_COMMON_H_ */
