"""The steady state of the matrix-core product of the direct correlator:
sizes whose splits hold several pairs of full source stages (off-diagonal
tiles with all four sub-tiles live), an odd and an even number of pairs, with
partial sums and with a single split that writes vis itself, every precision
and both phase conventions, against the FP64 product of the same inputs.

Tolerance: as in test_xcorr_product_gpu: a value is a sum of T products (16
per source for matrices, 4 for scalars), each rounded at most T times, T of
one stage of at most 32 sources in FP32 (stages are added in FP64) and of all
sources in FP64: 2 T u sum |J| |B| |J|, and the last rounding to vis.
"""
import math

import numpy as np
import pytest

from gpu_util import gpu_cross_correlate
from test_xcorr_gpu import random_sky
from test_xcorr_product_gpu import rounded

pytestmark = pytest.mark.gpu


def launch(prec, matrix, ns, nsrc):
    """(splits, pairs of full stages in a whole split) by the launch rule:
    stages of 8 (FP64) or 16 k-steps, one source of matrices or two scalars
    each; tiles of 32 or 64 stations; splits by sqrt(stages / (0.026 tiles));
    a pair starts while three whole stages are left."""
    tile = (8 if prec == "d" else 16) * (1 if matrix else 2)
    st = 32 if matrix else 64
    nb = -(-ns // st)
    stages = -(-nsrc // tile)
    assert nb >= 2 and ns >= 2 * st          # a full off-diagonal tile
    tiles = nb * (nb + 1) // 2
    splits = max(1, int(math.sqrt(stages / (0.026 * tiles))))
    per = -(-stages // splits)
    whole = min(per, nsrc // tile)
    return -(-stages // per), max(0, (whole - 1) // 2)


def product(g, ns, nsrc, matrix, casa):
    """V and the sum of magnitudes of every baseline, FP64."""
    q, p = np.triu_indices(ns, 1)
    if not matrix:
        j = g["jones_s"].reshape(ns, nsrc, 2)
        a = np.abs(j).sum(-1)
        j = j[..., 0] + 1j * j[..., 1]
        v = (j * g["I"]) @ j.conj().T
        mag = (a * np.abs(g["I"])) @ a.T
        v = v[q, p] if casa else v[p, q]
        return np.stack([v.real, v.imag], -1), mag[p, q][:, None]
    j = g["jones_m"].reshape(ns, nsrc, 2, 2, 2)
    a = np.abs(j).sum(-1)
    j = j[..., 0] + 1j * j[..., 1]
    i, qq, u, v = (g[k] for k in "IQUV")
    b = np.stack([i + qq, u + 1j * v, u - 1j * v, i - qq], -1).reshape(
        -1, 2, 2)
    m = np.stack([np.abs(i) + np.abs(qq), np.abs(u) + np.abs(v)] * 2, -1)
    m = m[:, [0, 1, 1, 0]].reshape(-1, 2, 2)

    def whole(left, right):
        x = np.matmul(left, right[0]).transpose(0, 2, 1, 3).reshape(
            2 * ns, -1)
        y = right[1].transpose(0, 2, 1, 3).reshape(2 * ns, -1)
        return (x @ y.conj().T).reshape(ns, 2, ns, 2)

    full, mag = whole(j, (b, j)), whole(a, (m, a))
    first, second = (q, p) if casa else (p, q)
    full = full[first, :, second, :].reshape(-1, 4)
    return np.stack([full.real, full.imag], -1).reshape(-1, 8), \
        mag[first, :, second, :].reshape(-1, 4).repeat(2, -1)


# precision, matrix, stations, sources -> splits, pairs
SIZES = [
    ("f", 1, 200, 5000, 20, 7), ("f", 1, 193, 6001, 21, 8),
    ("d", 1, 200, 2500, 20, 7), ("d", 1, 193, 3001, 21, 8),
    ("f", 0, 320, 9600, 25, 5), ("f", 0, 330, 7001, 20, 5),
    ("d", 0, 320, 4800, 25, 5), ("d", 0, 330, 3500, 20, 5),
    ("f", 0, 130, 6016, 32, 2), ("d", 0, 128, 6001, 63, 2),
    # one split
    ("f", 1, 512, 208, 1, 6), ("d", 1, 512, 104, 1, 6),
    ("f", 1, 520, 131, 1, 3), ("d", 1, 520, 65, 1, 3),
    ("f", 0, 512, 96, 1, 1), ("d", 0, 512, 48, 1, 1),
    ("f", 0, 1024, 416, 1, 6), ("d", 0, 1030, 171, 1, 4)]


@pytest.mark.parametrize("prec,matrix,ns,nsrc,splits,pairs", SIZES)
def test_pairs_of_stages(hip, prec, matrix, ns, nsrc, splits, pairs):
    assert launch(prec, matrix, ns, nsrc) == (splits, pairs)
    print(prec, matrix, ns, nsrc, flush=True)
    g = rounded(random_sky(np.random.default_rng(ns + nsrc), ns, nsrc), prec)
    u = 2.0 ** (-53 if prec == "d" else -24)
    nr = 8 if matrix else 2
    for casa in (0, 1):
        init = rounded(dict(v=np.random.default_rng(1).normal(
            size=ns * (ns - 1) // 2 * nr)), prec)["v"]
        got = gpu_cross_correlate(prec, casa, 0, matrix, g, 0, 0,
                                  vis_init=init).reshape(-1, nr)
        want, mag = product(g, ns, nsrc, matrix, casa)
        t = (16 if matrix else 4) * (nsrc if prec == "d" else 32) + 8
        err = np.abs(got - init.reshape(-1, nr) - want)
        tol = 2 * t * u * mag + 2 * u * (np.abs(init.reshape(-1, nr)) +
                                         np.abs(want))
        assert np.all(err <= tol), np.max(err / tol)


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("matrix", [0, 1])
@pytest.mark.parametrize("ns,nsrc", [(2, 20001), (5, 6007), (17, 6007),
                                     (33, 5003), (64, 3001), (65, 3001),
                                     (96, 2500), (97, 2500)])
def test_many_splits_of_few_stations(hip, prec, matrix, ns, nsrc):
    """Up to three tiles: hundreds of splits, each the sum of up to four
    waves, added by 16 waves; more tiles by four.  (Scalars of up to 32
    stations take the per-baseline kernel.)"""
    g = rounded(random_sky(np.random.default_rng(ns + nsrc), ns, nsrc), prec)
    u = 2.0 ** (-53 if prec == "d" else -24)
    nr = 8 if matrix else 2
    for casa in (0, 1):
        got = gpu_cross_correlate(prec, casa, 0, matrix, g, 0, 0).reshape(
            -1, nr)
        want, mag = product(g, ns, nsrc, matrix, casa)
        t = (16 if matrix else 4) * (nsrc if prec == "d" else 32) + 8
        err = np.abs(got - want)
        tol = 2 * t * u * mag + 2 * u * np.abs(want)
        assert np.all(err <= tol), np.max(err / tol)
