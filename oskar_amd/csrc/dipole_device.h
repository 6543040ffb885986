/*
 * Device functions of the dipole element pattern, shared by the pattern
 * kernels (beam_util.hip) and the aperture-array beam (dftw.hip): theta and
 * phi of an ENU direction
 * (oskar/convert/define_convert_enu_directions_to_theta_phi.h) and the
 * pattern of a pair of crossed dipoles
 * (oskar/telescope/station/element/define_evaluate_dipole_pattern.h).
 */
#ifndef OSKAR_AMD_DIPOLE_DEVICE_H_
#define OSKAR_AMD_DIPOLE_DEVICE_H_

#include "device_common.h"

namespace oskar_amd {

/* theta and the two phi (each offset by its delta, in [0, 2 pi)) of one
 * ENU direction. */
template <typename FP>
__device__ __forceinline__ void theta_phi_point(FP xx, FP yy, FP zz,
        FP delta_phi1, FP delta_phi2, FP* theta, FP* phi1, FP* phi2)
{
    const FP twopi = 2 * pi_v<FP>();
    const FP p0 = atan2(yy, xx);
    FP p1 = fmod(p0 + delta_phi1, twopi);
    FP p2 = fmod(p0 + delta_phi2, twopi);
    if (p1 < (FP) 0) p1 += twopi;
    if (p2 < (FP) 0) p2 += twopi;
    *theta = atan2(sqrt(xx * xx + yy * yy), zz);
    *phi1 = p1;
    *phi2 = p2;
}

/* One dipole: E_theta, E_phi (imaginary parts zero). */
template <typename FP>
__device__ __forceinline__ void dipole(FP phi, FP sin_theta, FP cos_theta,
        FP kL, FP cos_kL, Cplx<FP>* e_theta, Cplx<FP>* e_phi)
{
    FP sin_phi, cos_phi;
    sincos_v<FP>(phi, &sin_phi, &cos_phi);
    const FP denom = (FP) 1 + cos_phi * cos_phi * (cos_theta * cos_theta -
            (FP) 1);
    e_theta->y = e_phi->y = (FP) 0;
    if (denom == (FP) 0)
    {
        e_theta->x = e_phi->x = (FP) 0;
    }
    else
    {
        const FP t = (cos(kL * cos_phi * sin_theta) - cos_kL) / denom;
        e_theta->x = -cos_phi * cos_theta * t;
        e_phi->x = sin_phi * t;
    }
}

/* The dipole pattern of one direction, written to pattern[o]: the 2x2
 * matrix (X theta, X phi; Y theta, Y phi), rows swapped with swap_xy, or
 * for a scalar pattern the amplitude sqrt(sum of squares / 2). */
template <typename FP, bool MATRIX>
__device__ __forceinline__ void dipole_point(FP theta, FP phi_x, FP phi_y,
        FP kL, FP cos_kL, int swap_xy, Cplx<FP>* pattern, size_t o)
{
    FP sin_theta, cos_theta;
    sincos_v<FP>(theta, &sin_theta, &cos_theta);
    Cplx<FP> x_th, x_ph, y_th, y_ph;
    dipole<FP>(phi_x, sin_theta, cos_theta, kL, cos_kL, &x_th, &x_ph);
    dipole<FP>(phi_y, sin_theta, cos_theta, kL, cos_kL, &y_th, &y_ph);
    if (MATRIX)
    {
        Cplx<FP>* p = pattern + 4 * o;
        if (swap_xy)
        {
            p[0] = y_th; p[1] = y_ph; p[2] = x_th; p[3] = x_ph;
        }
        else
        {
            p[0] = x_th; p[1] = x_ph; p[2] = y_th; p[3] = y_ph;
        }
    }
    else
    {
        const FP amp = sqrt((x_th.x * x_th.x + x_ph.x * x_ph.x +
                y_th.x * y_th.x + y_ph.x * y_ph.x) / (FP) 2);
        pattern[o].x = amp;
        pattern[o].y = (FP) 0;
    }
}

/* The dipole pattern of one ENU direction from its coordinates: the same
 * as theta_phi_point then dipole_point, with the sines and cosines of theta
 * and phi as quotients of the coordinates (phi = 0 or pi at the zenith, as
 * atan2) and each feed's phi turned by its delta's sine and cosine (the
 * angles took two atan2, two fmod and three sincos per direction). */
template <typename FP> struct DipoleParams
{
    FP kL, cos_dx, sin_dx, cos_dy, sin_dy;
    int swap_xy;
};

template <typename FP, bool MATRIX>
__device__ __forceinline__ void dipole_enu_point(FP x, FP y, FP z,
        const DipoleParams<FP>& P, Cplx<FP>* pattern, size_t o)
{
    /* inv_sqrt and quotient take normal numbers.  Directions next to the
     * zenith, whose x^2 + y^2 is below TINY, are scaled up for phi (theta is
     * 0 there), so far that the least subnormal has a normal square; vectors
     * that are that short altogether are scaled as a whole. */
    constexpr FP TINY = sizeof(FP) == 4 ? (FP) 1e-30 : (FP) 1e-280;
    constexpr FP UP = sizeof(FP) == 4 ? (FP) 0x1p100 : (FP) 0x1p800;
    FP r2 = x * x + y * y;
    FP h2 = r2 + z * z;
    const bool up = r2 < TINY, is_short = h2 < TINY;
    const FP ux = up ? x * UP : x, uy = up ? y * UP : y;
    const FP uz = is_short ? z * UP : z;
    r2 = ux * ux + uy * uy;
    if (is_short) h2 = r2 + uz * uz;
    const bool zenith = !(r2 > (FP) 0);
    const FP ir = inv_sqrt(r2), ih = inv_sqrt(h2);
    const FP cos_theta = h2 > (FP) 0 ? uz * ih : (FP) 1;
    const FP sin_theta = r2 == (FP) 0 || up != is_short ? (FP) 0 :
            r2 * ir * ih;
    const FP cos_phi = zenith ? copysign((FP) 1, x) : ux * ir;
    const FP sin_phi = zenith ? (FP) 0 : uy * ir;
    FP e[2][2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
    {
        const FP cd = k ? P.cos_dy : P.cos_dx, sd = k ? P.sin_dy : P.sin_dx;
        const FP c = cos_phi * cd - sin_phi * sd;
        const FP s = sin_phi * cd + cos_phi * sd;
        /* t = (cos(kL q) - cos(kL)) / (1 - q^2), q = cos(phi) sin(theta),
         * with no difference of nearly equal values: 1 - q^2 as the sum of
         * the other coordinates' squares, and the numerator as 2 sin(kL (1 +
         * |q|) / 2) sin(kL (1 - |q|) / 2).  The first angle is rounded, so
         * next to the nulls of dipoles of kL = pi and more, where its sine is
         * near zero, the error is that of the angle, not of the value. */
        const FP q = fabs(c) * sin_theta, sy = s * sin_theta;
        const FP denom = fma(sy, sy, cos_theta * cos_theta);
        const FP half = (FP) 0.5 * P.kL;
        const FP up_q = (FP) 1 + q;
        const FP num = sin_fold(half * up_q) *
                sin_fold(half * quotient(denom, up_q));
        /* Along the dipole's axis (denom = sin^2 of the angle to it), where
         * t stays finite and the field goes to zero: zero. */
        const FP t = denom < TINY ? (FP) 0 : (FP) 2 * quotient(num, denom);
        e[k][0] = -c * cos_theta * t;
        e[k][1] = s * t;
    }
    const int row = MATRIX && P.swap_xy ? 1 : 0;
    if (MATRIX)
    {
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            Cplx<FP> v;
            v.x = row ? e[1 - k / 2][k % 2] : e[k / 2][k % 2];
            v.y = (FP) 0;
            pattern[4 * o + k] = v;
        }
    }
    else
    {
        Cplx<FP> v;
        v.x = sqrt((e[0][0] * e[0][0] + e[0][1] * e[0][1] +
                e[1][0] * e[1][0] + e[1][1] * e[1][1]) / (FP) 2);
        v.y = (FP) 0;
        pattern[o] = v;
    }
}

} /* namespace oskar_amd */

#endif /* OSKAR_AMD_DIPOLE_DEVICE_H_ */
