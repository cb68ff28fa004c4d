"""FP64 Green-Kubo calls with segments on one series at the same time: from
several threads, on several streams, and captured into a graph that is replayed
after larger calls.  Every result equals the call's own on a fresh series."""
import ctypes
import threading

import numpy as np
import pytest

from analisi_amd import capi, synth

pytestmark = pytest.mark.gpu

IDX = np.array([0, 3], np.uint32)


def _alone(J, tmax, n_seg, primo, n):
    return capi.DeviceSeries(J).gk_blocks([0, 3], 1, tmax, n_seg, True, tmax // 2, primo, n)


def test_threads():
    J = synth.ar2_currents(11, 9000)
    calls = [(40, 4, [0, 10], [200, 200]), (700, 4, [0, 500, 900], [2000] * 3), (1500, 7, [100, 300], [3000, 3100]),
             (65, 3, [5] * 20, [333] * 20)]
    want = [_alone(J, *c) for c in calls]
    s = capi.DeviceSeries(J)
    errors = []

    def work(k):
        try:
            tmax, n_seg, primo, n = calls[k]
            for _ in range(8):
                got = s.gk_blocks([0, 3], 1, tmax, n_seg, True, tmax // 2, primo, n)
                for a, b in zip(got, want[k]):
                    assert np.array_equal(a, b, equal_nan=True)
                one = s.gk([0, 3], 1, tmax, n[0], n_seg, True, tmax // 2, primo[0])
                assert np.array_equal(one, want[k][0][0], equal_nan=True)
        except BaseException as e:
            errors.append((k, e))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(calls))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors


class _Hip:
    def __init__(self):
        self.h = ctypes.CDLL("libamdhip64.so")

    def __call__(self, name, *a):
        assert getattr(self.h, name)(*a) == 0, name


def _async(s, out, tmax, n_seg, n, stream):
    p, k = np.zeros(1, np.uint64), np.full(1, n, np.uint32)
    capi.check(capi.lib().anl_gk_calculate_blocks_async(s.handle, capi._ptr(IDX), 2, 1, tmax, n_seg, 1, tmax // 2,
                                                        capi._ptr(p), capi._ptr(k), 1, capi.GK_FP64, out, None, None,
                                                        stream))


def test_streams():
    hip = _Hip()
    J = synth.ar2_currents(12, 9000)
    calls = [(1500, 4, 4000), (50, 5, 300), (900, 2, 2500)]
    want = [capi.DeviceSeries(J).gk([0, 3], 1, t, n, g, True, t // 2, 0) for t, g, n in calls]
    s = capi.DeviceSeries(J)
    streams = [ctypes.c_void_p() for _ in calls]
    for st in streams:
        hip("hipStreamCreateWithFlags", ctypes.byref(st), 1)
    outs = [[capi.DeviceBuffer(t * 14 * 8) for _ in range(6)] for t, _, _ in calls]
    for r in range(6):
        for c, st, o in zip(calls, streams, outs):
            _async(s, o[r].ptr, *c, st)
    for (t, _, _), st, o, w in zip(calls, streams, outs, want):
        hip("hipStreamSynchronize", st)
        for b in o:
            assert np.array_equal(b.to_host((t, 14)), w, equal_nan=True)
        hip("hipStreamDestroy", st)


def test_captured_call_replayed_after_larger_ones():
    hip = _Hip()
    J = synth.ar2_currents(13, 9000)
    want = capi.DeviceSeries(J).gk([0, 3], 1, 300, 1200, 4, True, 150, 0)
    s = capi.DeviceSeries(J)
    st, graph, run = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    hip("hipStreamCreateWithFlags", ctypes.byref(st), 1)
    out, big = capi.DeviceBuffer(300 * 14 * 8), capi.DeviceBuffer(3000 * 14 * 8)
    _async(s, out.ptr, 300, 4, 1200, st)
    hip("hipStreamSynchronize", st)
    hip("hipStreamBeginCapture", st, 1)
    _async(s, out.ptr, 300, 4, 1200, st)
    hip("hipStreamEndCapture", st, ctypes.byref(graph))
    hip("hipGraphInstantiate", ctypes.byref(run), graph, None, None, ctypes.c_size_t(0))
    for k in range(4):
        hip("hipGraphLaunch", run, st)
        hip("hipStreamSynchronize", st)
        assert np.array_equal(out.to_host((300, 14)), want, equal_nan=True), k
        _async(s, big.ptr, 900 + 700 * k, 4, 4000, st)
        s.gk([0, 3], 1, 500 + 500 * k, 3000, 4, False, 0, 0)
        hip("hipStreamSynchronize", st)
    hip("hipGraphExecDestroy", run)
    hip("hipGraphDestroy", graph)
    hip("hipStreamDestroy", st)
