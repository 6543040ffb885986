"""The direct correlator for few sources and many stations: the list of
station blocks (both orders, up to 3,001 stations), one split and several, and
the kernels that a call takes by its numbers of sources and stations, against
the CPU oracle.

Tolerance: relative RMS over all baselines, 5 roundings of the precision per
factor and product (1e-5 single with factors of arguments of up to some
hundred radians, 1e-6 without; 1e-12 and 1e-14 double).
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
    tol = {"f": 1e-6, "d": 1e-14}[prec]
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
