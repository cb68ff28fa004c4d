"""Spherical densities at the edges of the kernels' loops, against the oracle
(1e-12 of the largest value, as everywhere for these densities): every lmax on
both sides of the two unrolled ranges, atom counts around the blocks of 64
slots, cells large enough that blocks are skipped, and neighbour lists from
empty to more than 64 long."""
import numpy as np
import pytest

from analisi_amd import capi, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _case(seed, N, L, tri):
    tilt = (2.0 * synth.uniform(seed, 7, 3) - 1.0) * 0.15 * L if tri else None
    box = synth.lammps_box(L, tilt) if tri else synth.lammps_box(L)
    pos = synth.random_walk(seed, N, 3, box, 0.8)
    ot = O.Traj(pos, synth.types_by_fraction(N, [0.6, 0.4]), np.tile(box, (3, 1)), tri)
    return ot, capi.DeviceTrajectory(ot.pos, ot.box, ot.type_id, ot.ntypes, ot.cm)


def _close(got, want):
    assert np.abs(got - want).max() <= 1e-12 * max(np.abs(want).max(), 1e-300)


@pytest.mark.parametrize("tri", [False, True])
@pytest.mark.parametrize("lmax", [1, 5, 6, 7, 9, 10])
def test_lmax(lmax, tri):
    ot, dt = _case(21, 130, 9.5, tri)
    rm = np.array([[0.5, 3.0], [0.7, 2.8], [0.4, 3.1], [0.6, 2.9]])
    _close(capi.DeviceSph(dt, rm, 2, lmax).snapshot(2), O.sph_density(ot, 2, rm, 2, lmax))
    spec = [(60, 3.2 ** 2, 0.0), (60, 3.4 ** 2, 0.0)]
    s = capi.DeviceSph(dt, rm, 2, lmax)
    s.set_neighbours(spec)
    _close(s.snapshot(2), O.sph_density_sann(ot, 2, spec, 2, lmax)[0])


@pytest.mark.parametrize("tri", [False, True])
@pytest.mark.parametrize("N,L", [(2, 5.0), (63, 7.0), (64, 7.0), (65, 7.0), (257, 30.0), (700, 21.0), (4200, 40.0)])
def test_blocks_and_lists(N, L, tri):
    """Cutoffs from a few neighbours to lists of more than 64 atoms."""
    ot, dt = _case(22, N, L, tri)
    rm = np.tile([0.5, 2.6], (4, 1))
    _close(capi.DeviceSph(dt, rm, 1, 4).snapshot(1), O.sph_density(ot, 1, rm, 1, 4))
    for cut in (1.0, 3.0, 5.5):
        spec = [(500, cut ** 2, 0.0), (500, (0.9 * cut) ** 2, 0.0)]
        s = capi.DeviceSph(dt, rm, 1, 4)
        s.set_neighbours(spec)
        _close(s.snapshot(1), O.sph_density_sann(ot, 1, spec, 1, 4)[0])


@pytest.mark.parametrize("tri", [False, True])
@pytest.mark.parametrize("N,lmax,ll", [(21, 1, [1]), (64, 10, [2, 10]), (65, 7, [7]), (150, 10, [4, 6, 9])])
def test_averaged_order_parameter(N, lmax, ll, tri):
    """One wavefront per item: l values of one to all entries of two per lane,
    item counts around the 64 of a workgroup."""
    ot, dt = _case(23, N, 7.0 if N < 100 else 9.0, tri)
    spec = [(200, 3.4 ** 2, 0.0), (200, 3.1 ** 2, 0.0)]
    s = capi.DeviceSph(dt, np.tile([0.5, 2.6], (4, 1)), 1, lmax)
    s.set_neighbours(spec)
    q = s.steinhardt(3, 1, 0, ll, 12, do_histogram=False, averaged=True)
    want = O.steinhardt_sann(ot, spec, lmax, 12, ll, 1, 3, 0, False, averaged=True)
    same_nan = np.isnan(q) == np.isnan(want)
    assert same_nan.all() and np.nanmax(np.abs(q - want)) <= 1e-12
    h = s.steinhardt(3, 1, 0, ll, 12, averaged=True)
    hw = O.steinhardt_sann(ot, spec, lmax, 12, ll, 1, 3, 0, True, averaged=True)
    np.testing.assert_allclose(h, hw, rtol=1e-13, atol=0)
