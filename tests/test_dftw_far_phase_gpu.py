"""FP64 phases of the DFT and of the aperture-array beam past the range of the
polynomial sine and cosine (2^50 radians): phases that are exact products,
against the library's sine and cosine of the same double.

Tolerance: k whole revolutions are taken off with two doubles of 2 pi, whose
rest is below 2^-105, so k times it is below 2^-107 |x|.  k is within 2^-53 of
x / 2 pi, so the first difference is at most 2^-53 |x|, and it and the second
are rounded by at most 2^-106 |x| together: 2^-105 |x| in all, to which the
rounding of the reduced angle and of the polynomials (3e-16) and of the sum
are added.
"""
import numpy as np
import pytest

from gpu_util import gpu_dftw
from oskar_amd import lib
from oskar_amd.mem import OSKAR_DOUBLE, OSKAR_GPU, Station
from test_station_beam_gpu import AZEL, ENU_DIR, StationWork, station_beam
from test_station_errors_gpu import analyse

pytestmark = pytest.mark.gpu


def phases():
    rng = np.random.default_rng(6)
    v = np.exp2(rng.uniform(40, 90, 700)) * rng.choice([-1, 1], 700)
    edge = np.array([2.0 ** e for e in (49, 50, 51, 52, 53, 60)])
    near = np.concatenate([edge, -edge, np.nextafter(edge, 0),
                           np.nextafter(edge, np.inf)])
    return np.concatenate([v, near, rng.uniform(-50, 50, 57)])


@pytest.mark.parametrize("num_in,typed", [(1, 0), (6, 0), (6, 1)])
def test_dftw(hip, num_in, typed):
    x = phases()
    one, zero = np.ones(num_in), np.zeros(num_in)
    w = np.stack([one, zero], 1).ravel()
    idx = np.arange(num_in, dtype=np.int32) % 2 if typed else np.zeros(
        num_in, np.int32)
    data = np.stack([np.ones(2 * x.size), np.zeros(2 * x.size)], 1).ravel()
    got = gpu_dftw("d", 0, 0, 1.0, w, one, zero, None, x,
                   np.zeros(x.size), None, idx,
                   data).reshape(-1, 2)
    want = np.stack([np.cos(x), np.sin(x)], 1)
    tol = 2.0 ** -105 * np.abs(x) + 3e-16 + 2.0 ** -53 * num_in
    assert np.all(np.abs(got - num_in * want) <= num_in * tol[:, None])


def test_dftw_of_any_size_is_bounded(hip):
    """Phases that no double of 2 pi reduces: a unit phasor all the same;
    those that are no number stay none."""
    x = np.array([1e35, -1e60, 1e200, 1.7e308, np.inf, -np.inf, np.nan])
    one, zero = np.ones(1), np.zeros(1)
    data = np.stack([np.ones(x.size), np.zeros(x.size)], 1).ravel()
    got = gpu_dftw("d", 0, 0, 1.0, np.array([1.0, 0.0]), one, zero, None, x,
                   np.zeros(x.size), None, None, data).reshape(-1, 2)
    assert np.all(np.abs(np.hypot(*got[:4].T) - 1) < 1e-15)
    assert not np.any(np.isfinite(got[4:]))


@pytest.mark.parametrize("weights", [0, 1])
def test_beam(hip, weights):
    """Elements as far out, by their true or by their measured positions:
    a normalised array of unit phasors is at most 1 in every direction."""
    rng = np.random.default_rng(9)
    ne, n = 300, 1500
    far = 1e17 * rng.uniform(-1, 1, (3, ne))
    far[2] = 0
    st = Station(OSKAR_DOUBLE, OSKAR_GPU, ne)
    st.set_coords(*([0 * far, far] if weights else [far, 0 * far]))
    analyse(st)
    lib.oskar_station_set_phase_centre(st.ptr, AZEL, 0.3, 1.2)
    lib.oskar_station_set_normalise_array_pattern(st.ptr, 1)
    lib.oskar_station_set_normalise_final_beam(st.ptr, 0)
    z, p = rng.uniform(0, 1, n), rng.uniform(0, 2 * np.pi, n)
    r = np.sqrt(1 - z * z)
    got = station_beam(st, StationWork(OSKAR_DOUBLE, OSKAR_GPU), ENU_DIR, n,
                       (r * np.cos(p), r * np.sin(p), z), (AZEL, 0.3, 1.2),
                       60000.25, 140e6)
    assert np.max(np.abs(got)) < 1.0 + 1e-12
