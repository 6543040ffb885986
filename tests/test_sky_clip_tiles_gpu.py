"""oskar_sky_horizon_clip at the edges of its tiles of 2048 sources, with
none and all of the sky kept, and past the 2048 tiles up to which the last
pass adds the tiles' counts itself: mask, indices, every kept row and its
valid-column counts against the oracle's mask, prefix sum and row copy, value
for value."""
import numpy as np
import pytest

import oracle
from oskar_amd import lib
from oskar_amd.mem import Sky
from test_sky_gpu import clip_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,num", [
    ("f", 1), ("d", 2047), ("f", 2048), ("d", 2049), ("f", 4096),
    ("d", 70001), ("f", 4_200_001)])
def test_tiles(hip, prec, num):
    sky_in, sky_out, cols, want, got_mask, got_idx = clip_case(
        prec, num, [(0.3, -0.5)], 4.4, num)
    assert np.array_equal(got_mask, want)
    assert np.array_equal(got_idx, oracle.prefix_sum(want))
    total = int(want.sum())
    assert sky_out.attr(Sky.NUM_SOURCES) == total
    dt = np.float64 if prec == "d" else np.float32
    keep = np.nonzero(want)[0]
    for t, values in cols:
        assert np.array_equal(sky_out.get_column(t), values.astype(dt)[keep])
    for r in sorted({0, total // 2, total - 1} if total else set()):
        for t in (1, 3, 0x13):
            assert lib.oskar_sky_num_valid_columns_of_type(
                sky_out.ptr, t, r) == \
                lib.oskar_sky_num_valid_columns_of_type(
                    sky_in.ptr, t, int(keep[r]))


@pytest.mark.parametrize("models", [[], [(0.3, -0.5), (3.4, 0.5)]])
def test_none_and_all(hip, models):
    """No station model keeps nothing; two at opposite points keep all but
    the sources on their common horizon."""
    num = 5000
    sky_in, sky_out, cols, want, got_mask, got_idx = clip_case(
        "d", num, models, 1.0, 7)
    assert np.array_equal(got_mask, want)
    assert np.array_equal(got_idx, oracle.prefix_sum(want))
    keep = np.nonzero(want)[0]
    assert keep.size == (0 if not models else keep.size)
    assert sky_out.attr(Sky.NUM_SOURCES) == keep.size
    for t, values in cols:
        assert np.array_equal(sky_out.get_column(t), values[keep])


def test_number_kept_over_many_calls(hip):
    """More calls than pinned words for the number kept, of different sizes
    and numbers: each call returns its own."""
    for k in range(70):
        sky_in, sky_out, cols, want, got_mask, got_idx = clip_case(
            "f", 100 + 37 * k, [(0.3, -0.5)], 0.1 * k, k)
        assert sky_out.attr(Sky.NUM_SOURCES) == int(want.sum())
