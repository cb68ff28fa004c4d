"""g(r,t) with more workgroups than a launch can hold (a shape of one t0 per
workgroup over 4,200 t0 and 4,200 lags): the counts of the default shape."""
import numpy as np
import pytest

from analisi_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("varying,form", [(False, 2), (False, 0), (True, 2)])
def test_ranges(varying, form):
    F, N = 8400, 10
    rng = np.random.default_rng(2)
    pos = rng.uniform(0, 10, (F, N, 3))
    box = np.tile(np.array([0, 0, 0, 5, 5, 5.0]), (F, 1))
    if varying:
        box[:, 3:] += 1e-4 * rng.uniform(0, 1, (F, 1))
    t = capi.DeviceTrajectory(pos, box, np.zeros(N, np.int32), 1)
    g = capi.DeviceGofrt(t, 0.0, 4.0, 4, 4200, 1, 1, form)
    g.reset(4200)
    want = g.calculate(0)
    assert want.sum() > 0.2 * 4200 ** 2 * N * N
    g.set_tuning(4, 1, 1, 0)
    assert np.array_equal(g.calculate(0), want)
    assert g.pair_stats()["all"] == 4200 ** 2 * N * N
