"""Calls whose partial sums stay in a buffer of the library, on two streams
at once and from two host threads: each result equals the call's own, bit for
bit."""
import ctypes as C
import threading

import numpy as np
import pytest

from gpu_util import sync_check
from oskar_amd import capi, lib
from oskar_amd.mem import (OSKAR_COMPLEX, OSKAR_GPU, OSKAR_MATRIX,
                           OSKAR_SINGLE, Jones, Mem, check_status)
from test_xcorr_seam_gpu import _stream_create, _stream_destroy

pytestmark = pytest.mark.gpu


class Acorr:
    def __init__(self, seed, ns, nsrc):
        rng = np.random.default_rng(seed)
        P = OSKAR_SINGLE
        mt = P | OSKAR_COMPLEX | OSKAR_MATRIX
        self.nsrc = nsrc
        self.jones = Jones(mt, OSKAR_GPU, ns, nsrc)
        self.jones.set(rng.normal(size=ns * nsrc * 8))
        self.flux = [Mem.from_numpy(rng.uniform(0.1, 2, nsrc), P)
                     for _ in range(4)]
        self.args = capi.MEMA(*[m.ptr for m in self.flux])
        self.vis = Mem(mt, OSKAR_GPU, ns)

    def clear(self):
        self.vis.clear()

    def run(self, status):
        lib.oskar_auto_correlate(self.nsrc, self.jones.ptr, self.args, 0,
                                 self.vis.ptr, C.byref(status))

    def result(self):
        return [self.vis.numpy()]


def make(which):
    return Acorr(1, 300, 20000), Acorr(2, 257, 30000)


def serial(calls, which):
    s, want = C.c_int(0), []
    for x in calls:
        x.clear()
        x.run(s)
        check_status(s, which)
        sync_check(which)
        want.append(x.result())
    return want


def same(calls, want):
    for x, w in zip(calls, want):
        for a, b in zip(x.result(), w):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("which", ["acorr"])
def test_two_streams(hip, which):
    calls = make(which)
    want = serial(calls, which)
    s = C.c_int(0)
    streams = [_stream_create(), _stream_create()]
    try:
        for _ in range(3):
            for x in calls:
                x.clear()
            sync_check("clear")
            for x, st in zip(calls, streams):
                lib.oskar_hip_set_stream(st)
                x.run(s)
            lib.oskar_hip_set_stream(None)
            check_status(s, which)
            sync_check(which)
            same(calls, want)
    finally:
        lib.oskar_hip_set_stream(None)
        for st in streams:
            _stream_destroy(st)


@pytest.mark.parametrize("which", ["acorr"])
@pytest.mark.parametrize("own", [0, 1])
def test_two_threads(hip, which, own):
    """Two host threads, each on a stream of its own or both on the null
    stream, 20 calls each."""
    calls = make(which)
    want = serial(calls, which)
    streams = [_stream_create() if own else None for _ in calls]
    status = [C.c_int(0) for _ in calls]
    wrong = []

    def work(k):
        lib.oskar_hip_set_stream(streams[k])
        for _ in range(20):
            calls[k].clear()
            calls[k].run(status[k])
            got = calls[k].result()
            if status[k].value or not all(
                    np.array_equal(a, b) for a, b in zip(got, want[k])):
                wrong.append(k)
                return

    try:
        threads = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong, [s.value for s in status]
    finally:
        sync_check(which)
        for st in streams:
            if st:
                _stream_destroy(st)
