"""oskar_evaluate_jones_E over ENU directions, where flat stations of one
dipole type are evaluated up to 16 to a launch: every row equals
oskar_station_beam of its model (a launch of one, pinned against the CPU
oracle) bit for bit, whatever it shared a launch with.  Telescopes of 19
models that mix planar and 3D arrays, normalised and plain beams, element
errors (weights formed apart), a beam below the horizon (zeros) and, in
FP32, a station whose phases pass the hardware's exact range for some
directions only; direction counts at the edges of a workgroup and of one and
two directions per thread.
"""
import ctypes as C

import numpy as np
import pytest

from gpu_util import sync_check
from oskar_amd import capi, lib
from oskar_amd.mem import (OSKAR_COMPLEX, OSKAR_DOUBLE, OSKAR_GPU,
                           OSKAR_MATRIX, OSKAR_SINGLE, Jones, Mem,
                           StationView, StationWork, Telescope, check_status)

pytestmark = pytest.mark.gpu
ENU_DIR, AZEL = 1, 4
FREQ, MJD = 140e6, 60000.25
NS = 19


def telescope(rng, P):
    tel = Telescope(P, OSKAR_GPU, NS)
    s = C.c_int(0)
    lib.oskar_telescope_resize_station_array(tel.ptr, NS, C.byref(s))
    lib.oskar_telescope_set_phase_centre(tel.ptr, AZEL, 0.3, 1.1)
    for k in range(NS):
        ne = 5 + 16 * k
        st = StationView(lib.oskar_telescope_station(tel.ptr, k), P)
        lib.oskar_station_resize(st.ptr, ne, C.byref(s))
        radius = 600.0 if k == 7 else 15.0
        r = radius * np.sqrt(rng.uniform(size=ne))
        t = rng.uniform(0, 2 * np.pi, ne)
        z = rng.uniform(-1, 1, ne) if k % 5 == 3 else np.zeros(ne)
        st.set_coords(np.stack([r * np.cos(t), r * np.sin(t), z]))
        lib.oskar_station_set_phase_centre(
            st.ptr, AZEL, 0.2 * k, -0.5 if k == 11 else 1.0)
        lib.oskar_station_set_normalise_final_beam(st.ptr, int(k < 12))
        lib.oskar_station_set_normalise_array_pattern(st.ptr, k % 2)
        lib.oskar_station_set_swap_xy(st.ptr, int(k % 3 == 0))
        if k == 5:
            for e in range(ne):
                lib.oskar_station_set_element_errors(
                    st.ptr, 0, e, 1.0 + 0.01 * e, 0.0, 0.02 * e, 0.0,
                    C.byref(s))
            lib.oskar_station_analyse(st.ptr, C.byref(C.c_int(0)),
                                      C.byref(s))
        check_status(s, "station model")
    return tel


@pytest.mark.parametrize("prec,matrix,n", [
    ("d", 1, 1), ("f", 1, 255), ("d", 0, 257), ("f", 0, 513), ("d", 1, 3001),
    ("f", 1, 70001)])
def test_rows_equal_station_beam(hip, prec, matrix, n):
    rng = np.random.default_rng(n)
    P = OSKAR_DOUBLE if prec == "d" else OSKAR_SINGLE
    jt = P | OSKAR_COMPLEX | (OSKAR_MATRIX if matrix else 0)
    tel = telescope(rng, P)
    az = rng.uniform(-np.pi, np.pi, n)
    el = rng.uniform(-0.2, np.pi / 2, n)
    el[0] = np.pi / 2                       # the zenith
    dirs = [Mem.from_numpy(a, P) for a in
            (np.cos(el) * np.sin(az), np.cos(el) * np.cos(az), np.sin(el))]
    work = StationWork(P, OSKAR_GPU)
    E = Jones(jt, OSKAR_GPU, NS, n)
    s = C.c_int(0)
    d3 = capi.MEM3(*[m.ptr for m in dirs])
    lib.oskar_evaluate_jones_E(E.ptr, ENU_DIR, n, d3, 0.0, 0.0, tel.ptr, 0,
                               MJD, MJD, FREQ, work.ptr, C.byref(s))
    check_status(s, "oskar_evaluate_jones_E")
    sync_check("oskar_evaluate_jones_E")
    got = E.mem.numpy().reshape(NS, n, -1)
    for k in range(NS):
        out = Mem(jt, OSKAR_GPU, n)
        lib.oskar_station_beam(
            lib.oskar_telescope_station(tel.ptr, k), work.ptr, ENU_DIR, n,
            d3, 0.0, 0.0, AZEL, 0.3, 1.1, 0, MJD, MJD, FREQ, 0, out.ptr,
            C.byref(s))
        check_status(s, "oskar_station_beam")
        want = out.numpy().reshape(n, -1)
        assert np.all(np.isfinite(want))
        assert np.array_equal(got[k], want), k
        assert np.any(got[k]) == (k != 11 and bool(np.any(el >= 0))), k
