"""The FP64 Green-Kubo form where a lag has few t0 (a thread per lag), against the
oracle bit for bit: lag counts around a wavefront, empty segments, segments of one
term, strides of the whole range and beyond it, one to four currents, and both
sides of the line to the other kernels."""
import numpy as np
import pytest

from analisi_amd import capi, synth
from oracle import oracle as O
from test_gpu_gk_chain import _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,tmax,skip,n_seg", [
    (1, 1, 1, 1), (3, 3, 1, 2), (5, 5, 1, 7), (31, 30, 1, 100), (64, 63, 500, 1), (64, 64, 64, 1), (65, 65, 33, 2),
    (300, 129, 300, 1), (300, 129, 301, 3), (1000, 70, 90, 100), (1000, 70, 4294967295, 1), (1000, 300, 4294967289, 4),
    (4000, 1000, 1000, 16), (8, 8, 1, 1), (12, 12, 1, 1), (16, 16, 1, 1), (600, 600, 100, 3)])
def test_sizes(n, tmax, skip, n_seg):
    for ncur in (1, 2, 3, 4):
        J = synth.ar2_currents(9, n + min(n, tmax) + 2, ncur=ncur)
        idx = [3 * k for k in range(ncur)]
        s = capi.DeviceSeries(J)
        got = s.gk(idx, skip, tmax, n, n_seg, False, 0, 2)
        _same(got, O.gk(J, idx, skip, tmax, False, 0, n_seg, n, 2), ncur)


def test_blocks_and_values():
    """Blocks of different starts in one call; zeros, constants, infinities and
    NaN among the currents."""
    J = synth.ar2_currents(10, 2000, ncur=2)
    J[100:140] = 0.0
    J[150:155, 0] = 1e300
    J[155, 1] = np.inf
    J[300, 2] = np.nan
    s = capi.DeviceSeries(J)
    primo = list(range(0, 1500, 23))
    per, _, _ = s.gk_blocks([0, 3], 40, 70, 2, False, 0, primo, [120] * len(primo))
    for b, p in enumerate(primo):
        ref = O.gk(J, [0, 3], 40, 70, False, 0, 2, 120, p)
        assert np.array_equal(per[b], ref, equal_nan=True), p
