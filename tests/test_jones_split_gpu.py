"""K in groups of stations sized by the launch, and joins of matrices with
scalars in 16-byte parts, at sizes where groups and parts end unevenly.

Tolerances: as in test_jones_gpu: K against FP64 of the same inputs within
4 eps of the phase's largest terms plus 1e-6 (FP32) or 1e-14 (FP64) for the
sine; joins bit for bit against numpy in the same precision."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import prec_code
from oskar_amd import lib
from oskar_amd.mem import (OSKAR_COMPLEX, OSKAR_GPU, OSKAR_MATRIX, Jones,
                           check_status)
from test_jones_gpu import C0, gpu_K, np_join_exact, rand_jones

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("ns,nsrc", [(5, 257), (101, 6001), (7, 99901),
                                     (19, 200001)])
def test_K_groups(hip, prec, ns, nsrc):
    print("K", prec, ns, nsrc, flush=True)
    rng = np.random.default_rng(ns)
    dt = np.float64 if prec == "d" else np.float32
    l, m = (0.2 * rng.uniform(-1, 1, (2, nsrc))).astype(dt)
    n = np.sqrt(1 - l.astype(np.float64) ** 2 - m ** 2).astype(dt)
    u, v, w = (100 * rng.normal(size=(3, ns))).astype(dt)
    filt = rng.uniform(0, 1, nsrc).astype(dt)
    freq = 1e8
    got = gpu_K(prec, ns, l, m, n, u, v, w, freq, filt, 0.1, 0.9)
    got = np.asarray(got, np.float64).reshape(-1).view(
        np.complex128).reshape(ns, nsrc)
    k = 2 * np.pi * freq / C0
    terms = [np.outer(a.astype(np.float64), b.astype(np.float64))
             for a, b in ((u, l), (v, m), (w, n.astype(dt) - dt(1)))]
    want = np.exp(1j * k * sum(terms))
    want *= (filt > dt(0.1)) & (filt <= dt(0.9))
    eps = 2.0 ** -52 if prec == "d" else 2.0 ** -23
    bound = 4 * eps * k * sum(np.abs(t) for t in terms) + (
        1e-14 if prec == "d" else 1e-6)
    assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("am", [0, 1])
@pytest.mark.parametrize("ns,nsrc", [(1, 1), (1, 255), (1, 257), (3, 1023)])
def test_join_parts(hip, prec, am, ns, nsrc):
    P = prec_code(prec)
    dt = np.float64 if prec == "d" else np.float32
    rng = np.random.default_rng(nsrc)
    a = rand_jones(rng, dt, am, ns, nsrc)
    b = rand_jones(rng, dt, 1 - am, ns, nsrc)
    mat = P | OSKAR_COMPLEX | OSKAR_MATRIX
    ta, tb = (mat, P | OSKAR_COMPLEX)[::1 if am else -1]
    J1, J2 = Jones(ta, OSKAR_GPU, ns, nsrc), Jones(tb, OSKAR_GPU, ns, nsrc)
    J1.set(a)
    J2.set(b)
    J3 = Jones(mat, OSKAR_GPU, ns, nsrc)
    s = C.c_int(0)
    for out in (J3, J1 if am else J2):
        lib.oskar_jones_join(out.ptr, J1.ptr, J2.ptr, C.byref(s))
        check_status(s, "oskar_jones_join")
        got = out.mem.numpy()
        assert np.array_equal(got, np_join_exact(a, b, am, 1 - am))
