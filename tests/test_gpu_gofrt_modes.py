"""The screen an untuned g(r,t) takes in a constant cell: the cluster screen
where far groups are skipped, the 16-bit screen where they cannot be.  Counts
equal the oracle's and those of every explicit mode on both sides of the line."""
import numpy as np
import pytest

from analisi_amd import capi, synth
from gpu_util import first_diff
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,L,rel,tilt,clustered", [
    (33, 8.0, 0.45, None, False), (64, 9.0, 0.3, [0.9, -0.7, 0.5], False), (1000, 32.0, 0.31, None, False),
    (1000, 32.0, 0.05, None, False), (6000, 60.0, 0.03, None, True), (6000, 60.0, 0.04, [5.0, -4.0, 3.0], True)])
def test_untuned_mode(N, L, rel, tilt, clustered):
    F, n, lags = 5, 2, 2
    box = synth.lammps_box(L, tilt)
    pos = synth.random_walk(11, N, F, box, 0.1)
    ot = O.Traj(pos, synth.types_by_fraction(N, [0.6, 0.4]), np.tile(box, (F, 1)), tilt is not None)
    dt = capi.DeviceTrajectory(ot.pos, ot.box, ot.type_id, ot.ntypes, ot.cm)
    ref, _ = O.gofrt(ot, 0.0, rel * L, 40, lags, 4, 1, 1, n, 0, want_vdata=False)
    for mode in (None, 0, 1, 2, 3, 4):
        g = capi.DeviceGofrt(dt, 0.0, rel * L, 40, lags)
        if mode is not None:
            g.set_tuning(8, 0, 1 << 30, mode)
        g.reset(n)
        got = g.calculate(0)
        assert first_diff(got, ref) is None, (mode, first_diff(got, ref))
        assert g.stats()[0] == capi.GOFRT_SCREENED
        if mode is None:
            assert (g.cluster_stats()[0] > 0) == clustered
