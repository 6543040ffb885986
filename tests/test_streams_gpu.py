"""Calls whose partial sums stay in a buffer of the library, on two streams
at once and from two host threads: each result equals the call's own, bit for
bit."""
import ctypes as C
import threading

import numpy as np
import pytest

from gpu_util import sync_check
from oskar_amd import capi, lib
from oskar_amd.mem import (OSKAR_COMPLEX, OSKAR_GPU, OSKAR_INT, OSKAR_MATRIX,
                           OSKAR_SINGLE, Jones, Mem, Sky, StationWork,
                           Telescope, check_status)
from test_sky_gpu import I_JY, SCRATCH_L, SCRATCH_M, SCRATCH_N, make_sky
from test_xcorr_seam_gpu import _hip, _stream_create, _stream_destroy

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


class Prefix:
    def __init__(self, seed, num):
        self.num = num
        self.src = Mem.from_numpy(np.random.default_rng(seed).integers(
            0, 9, num).astype(np.int32), OSKAR_INT)
        self.out = Mem(OSKAR_INT, OSKAR_GPU, num + 1)

    def clear(self):
        self.out.clear()

    def run(self, status):
        lib.oskar_prefix_sum(self.num, self.src.ptr, self.out.ptr,
                             C.byref(status))

    def result(self):
        return [self.out.numpy()]


class Clip:
    def __init__(self, seed, num):
        rng = np.random.default_rng(seed)
        P = OSKAR_SINGLE
        v = rng.normal(size=(3, num))
        v /= np.linalg.norm(v, axis=0)
        self.sky = make_sky(P, num, [
            (I_JY, rng.uniform(0.1, 9, num)), (SCRATCH_L, v[0]),
            (SCRATCH_M, v[1]), (SCRATCH_N, v[2])])
        self.sky.set_reference(1.1, -0.6)
        self.tel = Telescope(P, OSKAR_GPU, 4)
        s = C.c_int(0)
        lib.oskar_telescope_resize_station_array(self.tel.ptr, 1, C.byref(s))
        lib.oskar_station_set_position(
            lib.oskar_telescope_station(self.tel.ptr, 0), 0.3, -0.5, 0.0,
            0.0, 0.0, 0.0)
        self.out, self.work = Sky(P, OSKAR_GPU, 10), StationWork(P, OSKAR_GPU)

    def clear(self):
        pass

    def run(self, status):
        lib.oskar_sky_horizon_clip(self.out.ptr, self.sky.ptr, self.tel.ptr,
                                   0.8, self.work.ptr, C.byref(status))

    def result(self):
        return [np.array([self.out.attr(Sky.NUM_SOURCES)])] + [
            self.out.get_column(c) for c in (I_JY, SCRATCH_N)]


def make(which):
    if which == "acorr":
        return Acorr(1, 300, 20000), Acorr(2, 257, 30000)
    if which == "prefix_sum":
        return Prefix(1, 3000001), Prefix(2, 2500000)
    return Clip(1, 700001), Clip(2, 900000)


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


@pytest.mark.parametrize("which", ["acorr", "prefix_sum", "clip"])
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


@pytest.mark.parametrize("which", ["acorr", "prefix_sum", "clip"])
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


def test_more_streams_than_ever(hip):
    """1,100 streams, one after another: none is refused a buffer."""
    a = Acorr(3, 5, 300)
    want = serial([a], "acorr")
    s = C.c_int(0)
    streams = [_stream_create() for _ in range(1100)]
    try:
        for st in streams:
            a.clear()
            sync_check("clear")
            lib.oskar_hip_set_stream(st)
            a.run(s)
            check_status(s, "acorr")
            lib.oskar_hip_set_stream(None)
            sync_check("acorr")
        same([a], want)
    finally:
        lib.oskar_hip_set_stream(None)
        sync_check("acorr")
        for st in streams:
            _stream_destroy(st)


@pytest.mark.parametrize("which", ["acorr", "prefix_sum"])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_capture_on_a_new_stream(hip, which, mode):
    """A call warmed on the null stream is captured on a stream that has not
    run it (each capture mode); replays give the call's own result, also after
    a larger call."""
    x = Acorr(1, 60, 3000) if which == "acorr" else Prefix(1, 100001)
    larger = Acorr(2, 512, 9000) if which == "acorr" else Prefix(2, 5000001)
    want = serial([x], which)
    api, graph, run = _hip(), C.c_void_p(), C.c_void_p()
    s = C.c_int(0)
    stream = _stream_create()
    try:
        lib.oskar_hip_set_stream(stream)
        assert api.hipStreamBeginCapture(stream, mode) == 0
        x.run(s)
        assert api.hipStreamEndCapture(stream, C.byref(graph)) == 0
        check_status(s, which)
        assert api.hipGraphInstantiate(C.byref(run), graph, None, None,
                                       C.c_size_t(0)) == 0
        lib.oskar_hip_set_stream(None)
        for k in range(4):
            if k == 2:
                serial([larger], which)
            x.clear()
            sync_check("clear")
            assert api.hipGraphLaunch(run, stream) == 0
            assert api.hipStreamSynchronize(stream) == 0
            same([x], want)
    finally:
        lib.oskar_hip_set_stream(None)
        sync_check(which)
        _stream_destroy(stream)
