"""Green-Kubo blocks copied to the host through the ring of pinned pieces: the
values of each block's own calculation, for outputs below one piece, of exactly
and just over a few pieces, and larger than the ring, with and without the mean
and variance, on a new series and again on the same one."""
import numpy as np
import pytest

from analisi_amd import capi, synth

pytestmark = pytest.mark.gpu

PIECE = 2 << 20


@pytest.mark.parametrize("blocks,leff", [(2, 40), (2, PIECE // 40 // 2 + 1), (4, PIECE // 40), (5, PIECE // 40 + 7),
                                         (9, PIECE // 40 + 13)])
@pytest.mark.parametrize("stats", [False, True])
def test_values(blocks, leff, stats):
    n = leff
    J = synth.ar2_currents(7, blocks * 64 + n + leff, ncur=1)
    primo = [64 * b for b in range(blocks)]
    s = capi.DeviceSeries(J)
    # t0 stride n: one term per lag, so that long outputs are cheap
    one = [s.gk([0], n, leff, n, 1, False, 0, p) for p in primo]
    fresh = capi.DeviceSeries(J)
    for _ in range(3):
        got, mean, var = fresh.gk_blocks([0], n, leff, 1, False, 0, primo, [n] * blocks, stats=stats)
        for b in range(blocks):
            assert np.array_equal(got[b], one[b], equal_nan=True)
        if stats:
            np.testing.assert_allclose(mean, np.mean(one, axis=0), rtol=1e-9, atol=1e-12)
            assert var.shape == mean.shape and np.isfinite(var).all()
        else:
            assert mean is None and var is None
