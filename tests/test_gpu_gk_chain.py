"""The FP64 Green-Kubo kernels against the oracle, bit for bit, at the sizes
where their rounds, groups and paths meet: t0 counts around multiples of 16 and
48, t0 strides on both sides of the row layouts (1, 8 / 9, 64 / 65), segments,
blocks, launches past the chain kernel's share of the chip, and values whose
running means leave the range of the two-operation division (zeros, constants,
tiny and huge currents)."""
import numpy as np
import pytest

from analisi_amd import capi, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _same(got, ref, ncur):
    """Every column equal (NaN where NaN); the complements of 3 currents and
    more to 1e-9."""
    n = 3 * ncur * ncur
    k = slice(None) if ncur <= 2 else slice(0, n)
    bad = ~((got[:, k] == ref[:, k]) | (np.isnan(got[:, k]) & np.isnan(ref[:, k])))
    assert not bad.any(), "%d values differ, first at %s" % (bad.sum(), np.argwhere(bad)[0])
    if ncur > 2:
        np.testing.assert_allclose(got[1:, n:], ref[1:, n:], rtol=1e-9)


@pytest.mark.parametrize("n,tmax,skip,n_seg", [
    (1, 1, 1, 1), (15, 7, 1, 1), (16, 16, 1, 1), (17, 3, 1, 1), (47, 40, 1, 1), (48, 48, 1, 1), (49, 49, 1, 1),
    (95, 64, 1, 1), (96, 65, 1, 1), (97, 63, 1, 1), (145, 129, 1, 1), (200, 70, 1, 3), (333, 65, 1, 7), (5, 5, 1, 9),
    (190, 80, 2, 1), (401, 90, 3, 2), (257, 66, 8, 1), (300, 66, 9, 1), (900, 70, 20, 2), (1025, 64, 64, 1),
    (1300, 70, 65, 1), (2000, 30, 200, 1), (60, 10, 100, 1)])
def test_sizes(n, tmax, skip, n_seg):
    for ncur in (1, 2, 3):
        J = synth.ar2_currents(5, n + min(n, tmax) + 3, ncur=ncur)
        data = np.concatenate([np.ones((len(J), 1)), J], axis=1)
        idx = [1 + 3 * k for k in range(ncur)]
        s = capi.DeviceSeries(data)
        for primo in (0, 3):
            got = s.gk(idx, skip, tmax, n, n_seg, False, 0, primo)
            _same(got, O.gk(data, idx, skip, tmax, False, 0, n_seg, n, primo), ncur)


@pytest.mark.parametrize("start", [0, 100, 1023, 1199, 1200, 5000])
def test_mean_and_integral_tiles(start):
    """Lag counts of several scan tiles and a partial one, the mean taken from
    every place."""
    for ncur, tmax in ((1, 1200), (2, 1200), (3, 500), (4, 150)):
        J = synth.ar2_currents(6, 2600, ncur=ncur)
        idx = [3 * k for k in range(ncur)]
        got = capi.DeviceSeries(J).gk(idx, 1, tmax, 1300, 1, True, start, 0)
        _same(got, O.gk(J, idx, 1, tmax, True, start, 1, 1300, 0), ncur)


@pytest.mark.parametrize("ncur,blocks,tmax,n,n_seg", [(1, 64, 300, 301, 8), (1, 64, 257, 333, 7), (2, 40, 130, 147, 4),
                                                      (3, 16, 200, 211, 4), (4, 4, 1800, 1801, 1)])
def test_launches_that_fill_the_chip(ncur, blocks, tmax, n, n_seg):
    J = synth.ar2_currents(7, blocks * n + tmax, ncur=ncur)
    idx = [3 * k for k in range(ncur)]
    s = capi.DeviceSeries(J)
    primo = [b * n for b in range(blocks)]
    got, _, _ = s.gk_blocks(idx, 1, tmax, n_seg, False, 0, primo, [n] * blocks)
    for b in sorted({0, 1, blocks // 2, blocks - 1}):
        _same(got[b], O.gk(J, idx, 1, tmax, False, 0, n_seg, n, primo[b]), ncur)


@pytest.mark.parametrize("blocks", [1, 60])
@pytest.mark.parametrize("kind", ["zero", "constant", "sparse", "tiny", "denormal", "huge", "mixed", "nan"])
def test_values_outside_the_fast_division(kind, blocks):
    n, tmax = 150, 70
    rng = np.random.default_rng(11)
    J = rng.standard_normal((blocks * n + tmax, 6))
    if kind == "zero":
        J[:, 3:] = 0.0
    elif kind == "constant":
        J[:] = 0.1
    elif kind == "sparse":
        J[rng.random(J.shape) < 0.9] = 0.0
    elif kind == "tiny":
        J *= 2.0 ** -460
    elif kind == "denormal":
        J *= 2.0 ** -530
    elif kind == "huge":
        J *= 2.0 ** 512
    elif kind == "mixed":
        J *= 10.0 ** rng.uniform(-150, 150, J.shape)
    else:
        J[77, 1] = np.nan
        J[90, 4] = np.inf
    s = capi.DeviceSeries(J)
    primo = [b * n for b in range(blocks)]
    with np.errstate(all="ignore"):
        got, _, _ = s.gk_blocks([0, 3], 1, tmax, 9, False, 0, primo, [n] * blocks, stats=blocks > 1)
        for b in sorted({0, blocks - 1}):
            _same(got[b], O.gk(J, [0, 3], 1, tmax, False, 0, 9, n, primo[b]), 2)
        _same(s.gk([0, 3], 2, tmax, n, 1, True, 20, 0), O.gk(J, [0, 3], 2, tmax, True, 20, 1, n, 0), 2)
