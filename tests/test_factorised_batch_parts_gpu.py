"""Batches of many small units, which fill the chip at the configured part
size and keep it: their partial sums stay a fraction of a gigabyte, and the
units' visibilities match the FP64 oracle of the direct algorithm; batches of
a few, which take the one-call part sizes, equal the one call bit for bit."""
import ctypes as C

import numpy as np
import pytest

from fact_cases import make_case, oracle_direct, rounded
from gpu_util import sync_check
from helpers import rel_rms
from oskar_amd.mem import (OSKAR_COMPLEX, OSKAR_GPU, OSKAR_MATRIX,
                           OSKAR_SINGLE, FactorisedBatch, Mem, Telescope)
from test_factorised_gpu import run
from test_xcorr_seam_gpu import _hip

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert _hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("ns,nsrc,units,limit_mb", [
    (30, 2000, 4, 64), (30, 2000, 512, 256), (300, 500, 64, 256)])
def test_units(hip, ns, nsrc, units, limit_mb):
    P = OSKAR_SINGLE
    mt = P | OSKAR_COMPLEX | OSKAR_MATRIX
    c = make_case(ns + nsrc, ns, nsrc)
    flux = [Mem.from_numpy(c[k], P) for k in "IQUV"]
    dirs = [Mem.from_numpy(c[k], P) for k in "lmn"]
    uvw = [Mem.from_numpy(c[k], P) for k in "uvw"]
    beam = Mem.from_numpy(c["E"].ravel(), mt)
    nb = ns * (ns - 1) // 2
    vis = Mem(mt, OSKAR_GPU, units * nb)
    vis.clear()
    tel = Telescope(P, OSKAR_GPU, ns)
    batch = FactorisedBatch(P, 0, ns, units)
    freqs = [150e6, 140e6]
    for u in range(units):
        batch.set_unit(u, nsrc, beam, flux, dirs, uvw, freqs[u % 2], u * nb,
                       vis)
    sync_check("batch set up")
    free = free_bytes()
    batch.run(units, 0, tel)
    sync_check("batch")
    used = free - free_bytes()
    got = vis.numpy().reshape(units, -1)
    batch.free()
    assert used <= limit_mb << 20, used >> 20
    for k in (0, 1):
        one = run(c, "f", 0, freqs[k])
        want = oracle_direct(rounded(c, "f"), freqs[k])
        for u in (k, units - 2 + k):
            assert np.array_equal(got[u], got[k])
            assert rel_rms(got[u], want) < 1e-5
        if units < 8:
            assert np.array_equal(got[k], one)


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("ns,nsrc", [(300, 20), (1100, 60)])
def test_rows_of_few_parts(hip, prec, ns, nsrc):
    """One call of one part: rows of up to five workgroups, a baseline per
    thread (20 and 60 sources: 2e-5, as for other handfuls)."""
    c = make_case(ns + nsrc, ns, nsrc)
    want = oracle_direct(rounded(c, prec), 150e6)
    assert rel_rms(run(c, prec, 0, 150e6), want) < 2e-5
