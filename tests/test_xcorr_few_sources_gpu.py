"""The direct correlator for few sources and many stations: the list of
station blocks (both orders, up to 3,001 stations), one split and several, and
the kernels that a call takes by its numbers of sources and stations, against
the CPU oracle.

Tolerance: relative RMS over all baselines, 5 roundings of the precision per
factor and product (1e-5 single with factors of arguments of up to some
hundred radians, 1e-6 without; 1e-12 and 1e-14 double, and the square root of
the number of sources times its roundoff where that is more).
"""
import numpy as np
import pytest

from gpu_util import gpu_cross_correlate
from helpers import rel_rms
from test_xcorr_gpu import oracle_run, random_sky
from test_xcorr_product_gpu import rounded

pytestmark = pytest.mark.gpu


def compare(prec, casa, gauss, matrix, ns, nsrc, bs):
    print(prec, casa, gauss, matrix, ns, nsrc, bs, flush=True)
    g = rounded(random_sky(np.random.default_rng(ns + nsrc), ns, nsrc), prec)
    got = gpu_cross_correlate(prec, casa, gauss, matrix, g, bs, 0)
    want = oracle_run("d", casa, gauss, matrix, g, bs, 0)
    tol = {"f": 1e-6, "d": max(1e-14, nsrc ** 0.5 * 2.0 ** -53)}[prec]
    if gauss or bs:
        tol = {"f": 1e-5, "d": 1e-12}[prec]
    assert rel_rms(got, want) < tol


@pytest.mark.parametrize("casa", [0, 1])
@pytest.mark.parametrize("ns", [2, 31, 32, 33, 48, 49, 64, 65, 512, 529, 1025,
                                3001])
def test_station_blocks(hip, ns, casa):
    compare("d", casa, 1, 0, ns, 2 if ns > 2000 else 5, 0)


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("matrix", [0, 1])
@pytest.mark.parametrize("ns,nsrc", [(512, 20), (300, 33), (300, 100),
                                     (200, 64), (101, 131), (64, 33)])
def test_splits(hip, prec, matrix, ns, nsrc):
    """One split where its partial sums would cost more than they save,
    several with remainders otherwise."""
    compare(prec, ns % 2, 1, matrix, ns, nsrc, 1)


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("matrix,ns,nsrc", [
    (1, 513, 16), (1, 513, 17), (1, 512, 32), (1, 512, 33), (1, 3, 32),
    (0, 1024, 64), (0, 1025, 64), (0, 513, 65), (0, 512, 128), (0, 512, 129),
    (0, 2, 128), (0, 32, 65536), (0, 33, 6000), (0, 16, 66000),
    (0, 17, 66000)])
def test_kernel_of_few_sources(hip, prec, matrix, ns, nsrc):
    """Both sides of the rule that leaves few sources without factors to the
    per-baseline kernel."""
    for casa in (0, 1):
        compare(prec, casa, 0, matrix, ns, nsrc, 0)


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("matrix", [0, 1])
@pytest.mark.parametrize("ns", [2, 3, 8, 9, 16, 17, 31, 32, 33, 48, 49, 64,
                                65, 97, 128, 129])
def test_edges_of_the_product(hip, prec, matrix, ns):
    """The product's tiles and remainders of its stages, with more sources
    than the per-baseline kernel takes (scalars: from 33 stations)."""
    compare(prec, ns % 2, 0, matrix, ns, 129 + 5 * (ns % 13), 0)


@pytest.mark.parametrize("prec", ["f", "d"])
def test_infinite_scalars_of_the_product(hip, prec):
    """An infinite value in the last source (the one that pads a stage)
    leaves every baseline of the other stations unchanged."""
    ns, nsrc, bad = 50, 161, 20
    g = rounded(random_sky(np.random.default_rng(4), ns, nsrc), prec)
    want = gpu_cross_correlate(prec, 0, 0, 0, g, 0, 0).reshape(-1, 2)
    j = g["jones_s"].copy().reshape(ns, nsrc, 2)
    j[bad, -1, :] = np.inf
    g["jones_s"] = j.ravel()
    got = gpu_cross_correlate(prec, 0, 0, 0, g, 0, 0).reshape(-1, 2)
    q, p = np.triu_indices(ns, 1)
    other = (p != bad) & (q != bad)
    assert np.array_equal(got[other], want[other])
    assert not np.any(np.isfinite(got[~other]).all(axis=-1))
