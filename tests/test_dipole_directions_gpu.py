"""The dipole pattern of ENU directions where their coordinates leave the
normal floating-point range: next to the zenith (x and y from the least
subnormal to where x^2 + y^2 is exact), along a dipole's axis, and vectors so
short that their squares underflow.  One-element stations (array factor 1,
the aperture-array beam kernel) and stations of two orientations (the pattern
kernel), against the textbook dipole in extended precision.

Tolerance: each value is a product of a handful of rounded factors of at most
1 (16 roundings cover the kernel's longest chain), and t = 2 sin(a) sin(b) /
(1 - q^2), a + b = kL = pi / 2, is at most 1: 16 u.
"""
import ctypes as C

import numpy as np
import pytest

from gpu_util import sync_check
from oskar_amd import capi, lib
from oskar_amd.mem import (OSKAR_COMPLEX, OSKAR_DOUBLE, OSKAR_GPU,
                           OSKAR_MATRIX, OSKAR_SINGLE, Mem, Station,
                           StationWork, check_status)
from test_station_errors_gpu import analyse

pytestmark = pytest.mark.gpu
ENU_DIR, AZEL = 1, 4
FREQ, MJD, C0 = 140e6, 60000.25, 299792458.0


def pattern(x, y, z, angle, kL):
    """(n, 4) reals X theta, X phi, Y theta, Y phi for feeds turned by
    `angle`, in extended precision."""
    L = np.longdouble
    x, y, z = (np.asarray(a).astype(L) for a in (x, y, z))
    r, ph = np.hypot(x, y), np.arctan2(y, x)
    h = np.hypot(r, z)
    ct = np.where(h > 0, z / np.where(h > 0, h, 1), 1)
    st = np.where(h > 0, r / np.where(h > 0, h, 1), 0)
    out = []
    for turn in (-angle, np.pi / 2 - angle):
        c, s = np.cos(ph + L(turn)), np.sin(ph + L(turn))
        q, one = np.abs(c) * st, (s * st) ** 2 + ct ** 2
        safe = np.where(one > 0, one, 1)
        t = 2 * np.sin(L(kL) / 2 * (1 + q)) * np.sin(
            L(kL) / 2 * one / (1 + q)) / safe
        t = np.where(one > 0, t, 0)
        out += [-c * ct * t, s * t]
    return np.stack(out, -1)


def gpu_beam(prec, angles, x, y, z, length=None):
    """The matrix beam of dipoles at the origin, one per angle (degrees)."""
    P = OSKAR_DOUBLE if prec == "d" else OSKAR_SINGLE
    st = Station(P, OSKAR_GPU, len(angles))
    st.set_coords(np.zeros((3, len(angles))))
    s = C.c_int(0)
    for i, a in enumerate(angles):
        for feed in (0, 1):
            lib.oskar_station_set_element_feed_angle(
                st.ptr, feed, i, float(a), 0.0, 0.0, C.byref(s))
    if length is not None:
        lib.oskar_element_set_dipole_length(
            lib.oskar_station_element(st.ptr, 0), float(length),
            b"Wavelengths", C.byref(s))
    analyse(st)
    lib.oskar_station_set_phase_centre(st.ptr, AZEL, 0.0, np.pi / 2)
    lib.oskar_station_set_normalise_array_pattern(st.ptr, 0)
    lib.oskar_station_set_normalise_final_beam(st.ptr, 0)
    dt = np.float64 if prec == "d" else np.float32
    n = len(x)
    dirs = [Mem.from_numpy(np.asarray(a, dt), P) for a in (x, y, z)]
    out = Mem(P | OSKAR_COMPLEX | OSKAR_MATRIX, OSKAR_GPU, n)
    work = StationWork(P, OSKAR_GPU)
    lib.oskar_station_beam(
        st.ptr, work.ptr, ENU_DIR, n, capi.MEM3(*[m.ptr for m in dirs]),
        0.0, 0.0, AZEL, 0.0, np.pi / 2, 0, MJD, MJD, FREQ, 0, out.ptr,
        C.byref(s))
    check_status(s, "oskar_station_beam")
    sync_check("oskar_station_beam")
    got = out.numpy().reshape(n, 4, 2)
    return got[..., 0] + 1j * got[..., 1].astype(np.float64)


def directions(prec):
    if prec == "d":
        dt, small = np.float64, [5e-324, 1e-320, 1e-312, 3e-308, 4e-305,
                                 1e-290, 1e-170, 1e-150, 1e-140, 1e-130,
                                 1e-20, 1e-8]
        axis, short = [5e-324, 1e-300, 1e-160, 1e-140, 1e-18], 1e-170
    else:
        dt, small = np.float32, [1.4e-45, 3e-41, 5e-40, 9e-39, 2e-38, 9e-38,
                                 2e-37, 1e-30, 1e-20, 1e-16, 1e-15, 1e-14,
                                 1e-8]
        axis, short = [1.4e-45, 1e-40, 1e-20, 1e-15, 1e-9], 1e-25
    d = [(0, 0, 1), (0, 0, short)]
    for a in small:
        d += [(a, 0, 1), (0, -a, 1), (-a, 0.3 * a, 1), (0.5 * a, a, 1)]
    for a in axis:                     # the horizon along x and y
        d += [(1, 0, a), (-1, 0, a), (0, 1, a), (1, a, a)]
    for a in (0.6, 0.999):             # short vectors
        d += [(short * a, 0, short * np.sqrt(1 - a * a)),
              (short * a * 0.6, -short * a * 0.8,
               short * np.sqrt(1 - a * a))]
    return np.array(d).astype(dt).T


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("angles", [(0.0,), (25.0, -70.0)])
def test_directions_out_of_the_normal_range(hip, prec, angles):
    x, y, z = directions(prec)
    got = gpu_beam(prec, angles, x, y, z)
    want = sum(pattern(x, y, z, np.radians(a), np.pi / 2) for a in angles)
    bad = np.nonzero(~np.isfinite(got).all(-1))[0]
    assert bad.size == 0, [(x[i], y[i], z[i]) for i in bad[:4]]
    u = 2.0 ** (-53 if prec == "d" else -24)
    err = np.max(np.abs(got - want))
    assert err <= 16 * u * len(angles)


@pytest.mark.parametrize("prec", ["f", "d"])
def test_not_a_number_stays(hip, prec):
    """A direction with a coordinate that is no number has no beam."""
    x, y, z = np.full((3, 4), 0.5)
    x[1], y[2], z[3] = np.nan, np.nan, np.nan
    got = gpu_beam(prec, (0.0,), x, y, z)
    assert np.all(np.isfinite(got[0]))
    assert not np.any(np.isfinite(got[1:]).all(-1))


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("length", [0.1, 0.5, 1.0, 1.5, 2.0, 9.5])
def test_long_dipoles(hip, prec, length):
    """Dipoles of other lengths than half a wave, up to many sines of the
    pattern.  With denom = 1 - q^2 and q within 6 u, the angles a = kL (1 + q)
    / 2 and b = kL denom / (2 (1 + q)) are within 5 kL u and 4 kL u, so
    t = 2 sin(a) sin(b) / denom lies within
    2 u (5 kL |sin b| + 4 |sin a| min(kL, b)) / denom + 16 u |t|,
    |sin b| <= min(1, b); the sines' own 2.5 u are among the 16."""
    rng = np.random.default_rng(8)
    n, kL = 20000, np.pi * length
    dt = np.float64 if prec == "d" else np.float32
    z, p = rng.uniform(0, 1, n), rng.uniform(0, 2 * np.pi, n)
    r = np.sqrt(1 - z * z)
    x, y, z = (a.astype(dt) for a in (r * np.cos(p), r * np.sin(p), z))
    got = gpu_beam(prec, (0.0,), x, y, z, length)
    want = pattern(x, y, z, 0.0, kL)
    u = 2.0 ** (-53 if prec == "d" else -24)
    v = np.stack([x, y, z]).astype(np.float64)
    v /= np.linalg.norm(v, axis=0)
    for k in (0, 1):
        q = np.abs(v[k])
        denom = v[1 - k] ** 2 + v[2] ** 2
        a, b = kL / 2 * (1 + q), kL / 2 * denom / (1 + q)
        t = 2 * np.abs(np.sin(a) * np.sin(b)) / denom
        tol = 2 * u * (5 * kL * np.minimum(1, b) + 4 * np.abs(np.sin(a)) *
                       np.minimum(kL, b)) / denom + 16 * u * t
        err = np.abs(got[:, 2 * k:2 * k + 2] - want[:, 2 * k:2 * k + 2])
        assert np.all(err.max(-1) <= tol + 1e-300), (k, np.max(
            err.max(-1) / tol))
