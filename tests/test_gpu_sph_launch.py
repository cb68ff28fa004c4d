"""Order parameters over more (frame, atom) pairs than one launch can hold:
1,000 atoms x 68,000 frames, 50 frames repeated; the histograms of the 50."""
import numpy as np
import pytest

from analisi_amd import capi

pytestmark = pytest.mark.gpu


def test_many_frames():
    N, base, rep = 1000, 50, 1360
    rng = np.random.default_rng(4)
    L = 25.0
    pos = rng.uniform(0, L, (base, N, 3))
    box = np.tile(np.array([0, 0, 0, L / 2, L / 2, L / 2]), (base * rep, 1))

    def run(p):
        F = len(p)
        t = capi.DeviceTrajectory(p, box[:F], np.zeros(N, np.int32), 1)
        out = []
        for sann in (False, True):
            h = capi.DeviceSph(t, [(0.5, 3.0)], 1, 2)
            if sann:
                h.set_neighbours([(60, 16.0, 16.0)])
            for averaged in ([False, True] if sann else [False]):
                out.append(np.rint(h.steinhardt(F, 1, 0, [2], 16, averaged=averaged) * F))
        return out

    few = run(pos)
    many = run(np.tile(pos, (rep, 1, 1)))
    for a, b in zip(few, many):
        assert a.sum() > 0
        assert np.array_equal(a * rep, b)
