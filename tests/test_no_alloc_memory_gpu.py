"""The fixed array of oskar_cross_correlate_no_alloc, in a process of its own:
its memory is held only once the entry point has been called, and a first
call under stream capture (each capture mode) records a graph whose replays
give the direct call's visibilities."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))

MEMORY = """
import ctypes as C
import numpy as np
from gpu_util import gpu_cross_correlate
from test_xcorr_gpu import random_sky
from test_xcorr_seam_gpu import _hip

def used():
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert _hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return (total.value - free.value) >> 20

g = random_sky(np.random.default_rng(1), 20, 200)
for gauss, smear in ((0, 0), (1, 1)):
    before = used()
    gpu_cross_correlate("f", 0, gauss, 1, g, smear, smear)
before2 = used()
assert before2 - before < 64, (before, before2)
gpu_cross_correlate("f", 0, 1, 1, g, 1, 1,
                    entry="oskar_cross_correlate_no_alloc")
assert used() - before2 >= 256
"""

CAPTURE = """
import ctypes as C
import numpy as np
from gpu_util import sync_check
from oskar_amd import capi, lib
from oskar_amd.mem import check_status
from test_xcorr_seam_gpu import _direct, _direct_inputs, _hip, _stream_create
hip, mode = _hip(), %d
x = _direct_inputs(1, 64, 3000)
s = C.c_int(0)
x["vis"].clear()
_direct(x, s)                      # loads and warms the correlator
check_status(s, "direct")
sync_check("direct")
want = x["vis"].numpy()
assert np.any(want)
x["vis"].clear()
sync_check("clear")
stream, graph, run = _stream_create(), C.c_void_p(), C.c_void_p()
lib.oskar_hip_set_stream(stream)
assert hip.hipStreamBeginCapture(stream, mode) == 0
lib.oskar_cross_correlate_no_alloc(
    0, 0, x["nsrc"], x["jones"].ptr,
    capi.MEMA(*[m.ptr for m in x["flux"]]),
    capi.MEM3(*[m.ptr for m in x["dirs"]]),
    capi.MEM3(*[m.ptr for m in x["ext"]]), x["tel"].ptr,
    capi.MEM3(*[m.ptr for m in x["uvw"]]), 0.0, 150e6, 0, x["vis"].ptr,
    C.byref(s))
assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
check_status(s, "no_alloc under capture")
assert hip.hipGraphInstantiate(C.byref(run), graph, None, None,
                               C.c_size_t(0)) == 0
lib.oskar_hip_set_stream(None)
assert not np.any(x["vis"].numpy())
for _ in range(3):
    x["vis"].clear()
    sync_check("clear")
    assert hip.hipGraphLaunch(run, stream) == 0
    assert hip.hipStreamSynchronize(stream) == 0
    assert np.array_equal(x["vis"].numpy(), want)
"""


def child(code):
    env = dict(os.environ, PYTHONPATH=os.pathsep.join(
        [HERE, os.path.dirname(HERE)]))
    r = subprocess.run([sys.executable, "-c", code], env=env, timeout=100,
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-1500:]


def test_memory_is_held_only_after_a_call(hip):
    child(MEMORY)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_first_call_under_capture(hip, mode):
    child(CAPTURE % mode)
