"""Part sizes of the factorised correlators: calls with fewer workgroups
than the chip runs at once take smaller parts, others fill whole rounds, and
a batch takes the one-call sizes only while it leaves the chip idle.  Sizes
at the edges of the rule and of the 64-station tiles, the smallest included,
against the FP64 oracle of the direct algorithm (1e-5 relative RMS, the
factorised tolerance; 2e-5 below 64 sources, where a handful of products
averages nothing)."""
import numpy as np
import pytest

from fact_cases import (make_case, oracle_direct, oracle_direct_stations,
                        rounded, station_beams)
from helpers import rel_rms
from test_factorised_batch_gpu import BatchCase, UNITS, oracle_unit, tol
from test_factorised_gpu import run
from test_factorised_jones_gpu import f32
from test_factorised_jones_gpu import run as run_jones

pytestmark = pytest.mark.gpu
SIZES = [(2, 1), (3, 9), (63, 64), (64, 513), (65, 8192), (97, 12007),
         (129, 8193), (300, 4100)]


@pytest.mark.parametrize("ns,nsrc", SIZES)
def test_shared_beam(hip, ns, nsrc):
    c = make_case(ns + nsrc, ns, nsrc)
    want = oracle_direct(rounded(c, "f"), 150e6)
    assert rel_rms(run(c, "f", 0, 150e6), want) < (
        1e-5 if nsrc >= 64 else 2e-5)


@pytest.mark.parametrize("ns,nsrc", SIZES)
def test_beam_per_station(hip, ns, nsrc):
    c = make_case(ns + 7 * nsrc, ns, nsrc)
    E = station_beams(ns, ns, nsrc)
    want = oracle_direct_stations(rounded(c, "f"), f32(E), 150e6)
    assert rel_rms(run_jones(c, E, "f", 0, 150e6), want) < (
        1e-5 if nsrc >= 64 else 2e-5)


def test_full_batch_keeps_its_part_size(hip):
    """150 stations are 6 tiles, so parts of 128 sources make over 1,024
    work items of these units: the batch runs at that part size."""
    case = BatchCase("f", 0)
    case.batch.set_config(1, 128, 0, 1)
    assert 6 * sum(-(-u[0] // 128) for u in UNITS) >= 1024
    case.run()
    got = case.results()
    for u in range(len(UNITS)):
        if UNITS[u][0] == 0:
            assert not np.any(got[u])
        else:
            assert rel_rms(got[u], oracle_unit("f", u)) < tol(u)
