"""MSD launches at the edges of the rules that choose them: few lags per residue
in a launch that fills the chip (eight lags per thread), shapes chosen for other
strides, and more blocks than one launch can hold."""
import numpy as np
import pytest

from analisi_amd import capi
from gpu_util import make_case

pytestmark = pytest.mark.gpu


def _reference(x, types, nt, skip, tmax, n):
    out = np.empty((tmax, nt))
    for t in range(tmax):
        d = ((x[0:n:skip] - x[t:t + n:skip]) ** 2).sum(2).mean(0)
        out[t] = [d[types == k].mean() for k in range(nt)]
    return out


@pytest.mark.parametrize("tmax,n", [(11, 66), (33, 44), (33, 55), (9, 10)])
def test_few_lags_per_residue(tmax, n):
    """Both sides of the line, 50,000 atoms at stride 11; 1e-10 relative, the bound
    of every MSD kernel against the running mean."""
    ot, dt = make_case(41, 50000, 90, 75.0, [0.6, 0.4], 0.05)
    for cm in (False, True):
        x = ot.pos - ot.cm[:, ot.type_id] if cm else ot.pos
        got = capi.msd(dt, 11, tmax, False, cm, n, 0)
        np.testing.assert_allclose(got[:, 0], _reference(x, ot.type_id, 2, 11, tmax, n), rtol=1e-10, atol=0)


@pytest.mark.parametrize("N", [1, 64, 255, 257, 1000])
def test_both_kernels_same_bits(N):
    ot, dt = make_case(44, N, 60, 14.0, [0.5, 0.3, 0.2] if N > 2 else [1.0], 0.05)
    for skip, tmax, n in ((1, 7, 20), (4, 9, 30), (30, 30, 29)):
        for cm in (False, True):
            dt.set_msd_tile(16, 4)
            want = capi.msd(dt, skip, tmax, cm, cm, n, 1)
            dt.set_msd_tile(0)
            assert np.array_equal(capi.msd(dt, skip, tmax, cm, cm, n, 1), want), (skip, cm)


def test_chosen_shapes_at_strides():
    ot, dt = make_case(42, 700, 420, 18.0, [1.0], 0.05)
    calls = [(50, 200, 200), (3, 60, 200), (2, 200, 200), (1, 40, 200)]
    own = [capi.msd(dt, s, t, False, False, n, 0) for s, t, n in calls]
    for shape in dt.MSD_SHAPES[:-1]:
        dt.set_msd_tile(*shape)
        for (s, t, n), want in zip(calls, own):
            assert np.array_equal(capi.msd(dt, s, t, False, False, n, 0), want), (shape, s)


@pytest.mark.parametrize("skip", [1, 4])
def test_blocks_in_ranges(skip):
    """290,000 blocks of 240 values: finishing them takes more than 2^32 threads."""
    nb, n, nt = 290000, 4, 60
    ot, dt = make_case(43, 60, 12, 9.0, [1.0 / nt] * nt, 0.1)
    primo = [b % 5 for b in range(nb)]
    b = capi.DeviceBlocks(dt, primo, [n] * nb, msd=True, msd_skip=skip, msd_tmax=4, use_graph=False)
    b.run()
    per = b.msd_results()[2]
    for p in range(5):
        one = capi.msd(dt, skip, 4, False, False, n, p)
        assert (per[p::5] == one).all()
