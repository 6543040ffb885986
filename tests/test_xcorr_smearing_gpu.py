"""The smearing factors of the direct correlator by the size of their
argument: the polynomials for small and middling arguments, the reduced form
for large ones, their edges (1.6 and 4), arguments far past any array
(1e5, 1e12), and mixtures of extended and point sources.

One source and unit Jones values make every visibility the factor itself.
Reference: sin(x)/x and exp in FP64 numpy on the rounded inputs.  Tolerance:
the argument is three products and two sums in the precision (6 u |terms|,
and |d sinc/dx| <= min(1/2, 2/|x|)), the polynomials lie within 2.5 u of
sinc, and two factors and the accumulation add a few u; u is the unit
roundoff.
"""
import numpy as np
import pytest

from gpu_util import gpu_cross_correlate
from test_xcorr_product_gpu import rounded

pytestmark = pytest.mark.gpu
C0 = 299792458.0


def one_source(rng, ns, reach, matrix):
    """Bandwidth-smearing arguments spread over [0, reach]."""
    g = dict(u=np.linspace(0, 1, ns), v=np.zeros(ns), w=np.zeros(ns),
             x=np.zeros(ns), y=np.zeros(ns), l=np.array([0.5]),
             m=np.array([0.0]), n=np.array([np.sqrt(0.75)]),
             I=np.array([1.0]), Q=np.zeros(1), U=np.zeros(1), V=np.zeros(1),
             a=np.zeros(1), b=np.zeros(1), c=np.zeros(1))
    g["u"] = g["u"] + rng.uniform(0, 1e-3, ns)
    j = np.zeros((ns, 1, 8))
    j[..., 0] = j[..., 6] = 1.0
    g["jones_m"] = j.ravel()
    g["jones_s"] = np.tile([1.0, 0.0], ns)
    # pi (bw / f) (f / c) u l = reach at u = 1.
    bw = 2 * reach * C0 / np.pi
    g.update(freq=np.array(100e6), channel_bw=np.array(bw),
             time_avg=np.array(0.0), gast=np.array(0.0), ra0=np.array(0.0),
             dec0=np.array(0.0))
    return g


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("matrix", [0, 1])
@pytest.mark.parametrize("reach", [0.0, 1e-3, 1.0, 1.599, 1.601, 3.999,
                                   4.001, 12.0, 300.0, 1e5, 1.1e5, 2e10,
                                   1e12])
def test_sinc(hip, prec, matrix, reach):
    ns = 70
    g = rounded(one_source(np.random.default_rng(3), ns, reach, matrix), prec)
    got = gpu_cross_correlate(prec, 0, 0, matrix, g, 1, 0).astype(np.float64)
    got = got.reshape(-1, 8 if matrix else 2)[:, 0]
    u = 2.0 ** (-53 if prec == "d" else -24)
    q, p = np.triu_indices(ns, 1)
    dt = np.float64 if prec == "d" else np.float32
    f = float(g["freq"])
    frac = float(dt(float(g["channel_bw"]) / f))
    x = np.pi * frac * float(dt(f / C0)) * (g["u"][p] - g["u"][q]) * \
        g["l"][0]
    # n - 1 and m are zero or multiply zero coordinates.
    want = np.sinc(x / np.pi)
    slope = np.minimum(0.5, 2.0 / np.maximum(np.abs(x), 1e-300))
    tol = 6 * u * np.abs(x) * slope + 6 * u
    assert np.all(np.abs(got - want) <= tol), np.max(
        np.abs(got - want) / tol)


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("matrix", [0, 1])
def test_gaussian_and_point_sources_together(hip, prec, matrix):
    """Extended sources between point sources: the sum of the two skies
    correlated apart."""
    ns, nsrc = 45, 37
    rng = np.random.default_rng(8)
    from test_xcorr_gpu import random_sky
    g = random_sky(rng, ns, nsrc, spread=3000.0)
    ext = rng.uniform(size=nsrc) < 0.5
    for k in ("a", "b", "c"):
        g[k] = np.where(ext, g[k], 0.0)
    g = rounded(g, prec)
    nr = 8 if matrix else 2
    both = gpu_cross_correlate(prec, 0, 1, matrix, g, 1, 1)
    apart = np.zeros(both.size)
    for use in (ext, ~ext):
        h = dict(g)
        for k in ("I", "Q", "U", "V", "l", "m", "n", "a", "b", "c"):
            h[k] = g[k][use]
        h["jones_m"] = g["jones_m"].reshape(ns, nsrc, 8)[:, use].ravel()
        h["jones_s"] = g["jones_s"].reshape(ns, nsrc, 2)[:, use].ravel()
        apart += gpu_cross_correlate(prec, 0, 1 if use is ext else 0, matrix,
                                     h, 1, 1).astype(np.float64)
    u = 2.0 ** (-53 if prec == "d" else -24)
    j = np.abs(g["jones_m" if matrix else "jones_s"]).max()
    scale = (4 if matrix else 1) * 2 * j * j * 4.0 * nsrc
    assert np.max(np.abs(both - apart)) <= 16 * nr * u * scale


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("matrix", [0, 1])
@pytest.mark.parametrize("nsrc", [1, 3, 4, 5, 17, 65, 277])
def test_few_sources(hip, prec, matrix, nsrc):
    """Splits of fewer sources than a tile: the sum of each source on its
    own, to the rounding of a sum of nsrc terms."""
    ns = 30
    from test_xcorr_gpu import random_sky
    g = rounded(random_sky(np.random.default_rng(nsrc), ns, nsrc,
                           spread=3000.0), prec)
    nr = 8 if matrix else 2
    got = gpu_cross_correlate(prec, 0, 1, matrix, g, 1, 1)
    apart = np.zeros(got.size)
    for s in range(nsrc):
        h = dict(g)
        for k in ("I", "Q", "U", "V", "l", "m", "n", "a", "b", "c"):
            h[k] = g[k][s:s + 1]
        h["jones_m"] = g["jones_m"].reshape(ns, nsrc, 8)[:, s].ravel()
        h["jones_s"] = g["jones_s"].reshape(ns, nsrc, 2)[:, s].ravel()
        apart += gpu_cross_correlate(prec, 0, 1, matrix, h, 1,
                                     1).astype(np.float64)
    u = 2.0 ** (-53 if prec == "d" else -24)
    j = np.abs(g["jones_m" if matrix else "jones_s"]).max()
    scale = (4 if matrix else 1) * 2 * j * j * 4.0 * nsrc
    assert np.max(np.abs(got - apart)) <= 16 * nr * u * scale
