"""The direct correlator for point sources without smearing: sizes at the
edges of the matrix-core product's tiles (32 stations of matrices or 64 of
scalars per workgroup, halves of those per wave, 16 rows per MFMA block) and
of its source stages (8 or 16 k-steps), one split and many, and of the
per-baseline kernel, which takes up to 32 sources of matrices and 128 of
scalars on these arrays.  The product's pipeline (pairs of full stages) is in
test_xcorr_product_stages_gpu, its edges with more sources in
test_xcorr_few_sources_gpu.

Tolerance: a value is a sum of T products of reals (T = 16 per source for
matrices: 2 x 2 complex products on each of J B and M J^H; 4 for scalars),
each rounded at most T times, so it lies within 2 T u sum |J| |B| |J| of
the exact value, u the unit roundoff of the precision.  T <= 64 at most
counts for FP32, where a stage of sources is added to FP64 totals; the last
rounding to the output adds u |V|.
"""
import ctypes as C

import numpy as np
import pytest

from gpu_util import gpu_cross_correlate, sync_check
from oskar_amd import lib
from oskar_amd.mem import OSKAR_DOUBLE, OSKAR_SINGLE, Mem
from test_xcorr_gpu import oracle_run, random_sky

pytestmark = pytest.mark.gpu


def rounded(g, prec):
    dt = np.float64 if prec == "d" else np.float32
    keep = ("freq", "channel_bw", "time_avg", "gast", "ra0", "dec0")
    return {k: v if k in keep else v.astype(dt).astype(np.float64)
            for k, v in g.items()}


def bound(g, ns, nsrc, prec, matrix):
    """Elementwise bound on the rounding error of every output real."""
    u = 2.0 ** (-53 if prec == "d" else -24)
    if matrix:
        j = np.abs(g["jones_m"].reshape(ns, nsrc, 2, 2, 2)).sum(-1)
        i, q, uu, v = (np.abs(g[k]) for k in "IQUV")
        b = np.stack([i + q, uu + v, uu + v, i + q], -1).reshape(-1, 2, 2)
        mag = np.einsum("psik,skl,qsml->pqim", j, b, j)
    else:
        j = np.abs(g["jones_s"].reshape(ns, nsrc, 2)).sum(-1)
        mag = np.einsum("ps,s,qs->pq", j, np.abs(g["I"]), j)[..., None, None]
    q, p = np.triu_indices(ns, 1)
    terms = 16 if matrix else 4
    t = terms * (nsrc if prec == "d" else min(nsrc, 16)) + 8
    m = np.maximum(mag[p, q], mag[q, p].swapaxes(-1, -2))
    return (2 * t * u * m).reshape(q.size, -1).repeat(2, axis=-1)


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("matrix", [0, 1])
@pytest.mark.parametrize("ns,nsrc", [
    (2, 1), (8, 7), (9, 8), (16, 9), (17, 16), (31, 17), (32, 33), (33, 40),
    (48, 41), (49, 65), (64, 97), (65, 31), (97, 24), (130, 130), (33, 1500),
    (200, 5)])
def test_edges(hip, prec, matrix, ns, nsrc):
    rng = np.random.default_rng(ns * 1000 + nsrc)
    g = rounded(random_sky(rng, ns, nsrc), prec)
    casa = ns % 2
    print(prec, matrix, ns, nsrc, flush=True)
    got = gpu_cross_correlate(prec, casa, 0, matrix, g, 0, 0)
    want = oracle_run("d", casa, 0, matrix, g, 0, 0)
    err = np.abs(got.astype(np.float64) - want).reshape(
        -1, 8 if matrix else 2)
    tol = bound(g, ns, nsrc, prec, matrix)
    assert np.all(err <= tol), np.max(err / tol)


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("matrix", [0, 1])
def test_infinite_values_stay_with_their_station(hip, prec, matrix):
    """An infinite Jones value in the last source (the one that pads a
    stage) leaves every baseline of the other stations unchanged."""
    ns, nsrc, bad = 50, 61, 20
    rng = np.random.default_rng(4)
    g = rounded(random_sky(rng, ns, nsrc), prec)
    key = "jones_m" if matrix else "jones_s"
    nr = 8 if matrix else 2
    want = gpu_cross_correlate(prec, 0, 0, matrix, g, 0, 0).reshape(-1, nr)
    j = g[key].copy().reshape(ns, nsrc, nr)
    j[bad, -1, :] = np.inf
    g[key] = j.ravel()
    got = gpu_cross_correlate(prec, 0, 0, matrix, g, 0, 0).reshape(-1, nr)
    q, p = np.triu_indices(ns, 1)
    other = (p != bad) & (q != bad)
    assert np.array_equal(got[other], want[other])
    assert not np.any(np.isfinite(got[~other]).all(axis=-1))


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("matrix", [0, 1])
@pytest.mark.parametrize("nsrc", [30, 50, 150])
def test_jones_aligned_to_a_real_only(hip, prec, matrix, nsrc):
    """The raw-pointer entry points take Jones arrays with the alignment of
    one real, in both kernels."""
    ns = 40
    rng = np.random.default_rng(5)
    g = rounded(random_sky(rng, ns, nsrc), prec)
    P = OSKAR_DOUBLE if prec == "d" else OSKAR_SINGLE
    F = C.c_double if prec == "d" else C.c_float
    size = 8 if prec == "d" else 4
    nr = 8 if matrix else 2
    want = gpu_cross_correlate(prec, 0, 0, matrix, g, 0, 0)
    j = Mem.from_numpy(np.concatenate(
        [[0.0], g["jones_m" if matrix else "jones_s"]]), P)
    m = {k: Mem.from_numpy(g[k], P) for k in
         ("I", "Q", "U", "V", "l", "m", "n", "u", "v", "w", "x", "y")}
    vis = Mem.from_numpy(np.zeros(ns * (ns - 1) // 2 * nr), P)
    flux = ("I", "Q", "U", "V") if matrix else ("I",)
    name = "oskar_cross_correlate_%spoint_hip_%s" % (
        "" if matrix else "scalar_", prec)
    inv_wl = float(g["freq"]) / 299792458.0
    getattr(lib, name)(
        0, nsrc, ns, 0, C.c_void_p(j.data_ptr() + size),
        *[m[k].data_ptr() for k in flux],
        *[m[k].data_ptr() for k in ("l", "m", "n", "u", "v", "w", "x", "y")],
        F(0.0), F(3.4e38), F(inv_wl), F(0.0), F(0.0), F(0.0), F(0.0),
        vis.data_ptr())
    sync_check(name)
    assert np.array_equal(vis.numpy(), want)
