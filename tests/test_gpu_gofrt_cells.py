"""g(r,t) over a cell that changes along the trajectory (the automatic form
screens in each time origin's cell) against the oracle and the plain FP64
form: counts bit-exact.  Orthorhombic and triclinic cells, wrapped and far
unwrapped positions, sizes around the tiles of 256 and groups of 64 atoms, a
sparse large cell whose groups are skipped, skip and every, atom ranges,
blocks, pairs at bin edges, and the cases that stay with the plain form."""
import numpy as np
import pytest

from analisi_amd import capi, synth
from gpu_util import first_diff
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _case(seed, N, F, L, tilt, fractions=(0.5, 0.3, 0.2), shift=0.0, breathe=0.02):
    box0 = synth.lammps_box(L, tilt)
    pos = synth.random_walk(seed, N, F, box0, 0.15)
    rng = np.random.default_rng(seed)
    s = 1 + breathe * rng.uniform(-1, 1, (F, 3))
    box = np.tile(box0, (F, 1))
    box[:, [1, 3, 5]] *= s
    if tilt is not None:
        box[:, 6:] *= 1 + breathe * rng.uniform(-1, 1, (F, 3))
    pos *= s[:, None, :]
    if shift:
        pos[:, ::3] += shift
        pos[:, 1::7] -= 2.3 * shift
    ot = O.Traj(pos, synth.types_by_fraction(N, list(fractions)), box, tilt is not None)
    return ot, capi.DeviceTrajectory(ot.pos, ot.box, ot.type_id, ot.ntypes, ot.cm)


@pytest.mark.parametrize("N", [769, 831, 832, 1023, 1024, 1025])
@pytest.mark.parametrize("tilt,shift", [(None, 0.0), (None, 41.0), ([1.5, -1.2, 0.9], 0.0), ([-1.4, 1.1, 1.3], -37.0)])
def test_counts(N, tilt, shift):
    ot, dt = _case(5, N, 12, 17.0, tilt, shift=shift)
    for rmin, rmax, nbin, skip, every, n, primo in [(0.0, 6.5, 71, 1, 1, 6, 0), (0.4, 5.0, 40, 2, 2, 7, 1)]:
        ref, _ = O.gofrt(ot, rmin, rmax, nbin, 5, 8, skip, every, n, primo, want_vdata=False)
        g = capi.DeviceGofrt(dt, rmin, rmax, nbin, 5, skip, every)
        g.reset(n)
        got = g.calculate(primo)
        assert first_diff(got, ref) is None, first_diff(got, ref)
        st = g.pair_stats()
        assert g.stats()[0] == capi.GOFRT_SCREENED and g.stats()[1] >= ref.sum()
        assert st["screen16"] > 0 and st["fp64"] == 0 and st["all"] == N * N * -(-n // skip) * -(-5 // every)
        p = capi.DeviceGofrt(dt, rmin, rmax, nbin, 5, skip, every, capi.GOFRT_FP64)
        p.reset(n)
        assert np.array_equal(p.calculate(primo), got) and p.stats()[0] == capi.GOFRT_FP64


def test_far_groups_are_skipped():
    """4,000 atoms in a 60 A cell, rmax 5 A: most blocks of pairs are skipped,
    none that counts."""
    for tilt in (None, [6.0, -5.0, 4.0]):
        ot, dt = _case(6, 4000, 6, 60.0, tilt, shift=150.0)
        ref, _ = O.gofrt(ot, 0.0, 5.0, 50, 3, 8, 1, 1, 3, 0, want_vdata=False)
        g = capi.DeviceGofrt(dt, 0.0, 5.0, 50, 3)
        g.reset(3)
        got = g.calculate(0)
        assert first_diff(got, ref) is None, first_diff(got, ref)
        st = g.pair_stats()
        assert st["evaluated"] < 0.7 * st["all"]


def test_atom_ranges_and_blocks():
    ot, dt = _case(7, 800, 30, 16.0, [1.0, 0.8, -0.7])
    g = capi.DeviceGofrt(dt, 0.2, 6.0, 33, 6)
    g.reset(9)
    for t, im, a0, a1 in [(0, 0, 0, 800), (3, 5, 17, 18), (5, 2, 100, 333), (1, 8, 799, 800), (2, 1, 50, 50)]:
        c = np.zeros((6, 12, 33), np.uint64)
        O.gofrt_single(ot, 0.2, 6.0, 33, 6, t, im, a0, a1, 2, c)
        assert np.array_equal(g.calc_single_th(t, im, a0, a1, 2), c), (t, im, a0, a1)
    primo, n = [0, 7, 13], [7, 6, 11]
    eng = capi.DeviceBlocks(dt, primo, n, gofrt=g, use_graph=True)
    for _ in range(3):
        eng.run()
    counts = eng.gofrt_results()[2]
    for b in range(3):
        g.reset(n[b])
        assert np.array_equal(counts[b], g.calculate(primo[b]))


def test_pairs_at_bin_edges():
    """Pairs within ulps of every bin edge and of rmax, in a cell that differs
    from frame to frame."""
    rmax, nbin, N = 5.0, 25, 800
    rng = np.random.default_rng(8)
    box = np.tile(synth.lammps_box(14.0), (3, 1))
    box[1, 1] = 14.001
    box[2, 3] = 13.999
    pos = rng.uniform(0, 14, (3, N, 3))
    for k in range(N // 2):
        d = (k % (nbin + 1)) * (rmax / nbin)
        d = np.nextafter(d, [-np.inf, np.inf][k % 2]) if k % 3 else d
        pos[:, 2 * k + 1] = pos[:, 2 * k]
        pos[:, 2 * k + 1, k % 3] += d
    ot = O.Traj(pos, np.zeros(N, np.int32), box, False)
    dt = capi.DeviceTrajectory(ot.pos, ot.box, ot.type_id, ot.ntypes, ot.cm)
    ref, _ = O.gofrt(ot, 0.0, rmax, nbin, 2, 4, 1, 1, 2, 0, want_vdata=False)
    g = capi.DeviceGofrt(dt, 0.0, rmax, nbin, 2)
    g.reset(2)
    got = g.calculate(0)
    assert first_diff(got, ref) is None and g.stats()[0] == capi.GOFRT_SCREENED


def test_what_stays_with_the_plain_form():
    ot, dt = _case(9, 900, 8, 12.0, None)
    g = capi.DeviceGofrt(dt, 0.0, 6.2, 30, 2)       # over half of some frame's shortest edge
    g.reset(3)
    ref, _ = O.gofrt(ot, 0.0, 6.2, 30, 2, 4, 1, 1, 3, 0, want_vdata=False)
    assert np.array_equal(g.calculate(0), ref) and g.stats()[0] == capi.GOFRT_FP64
    s = capi.DeviceGofrt(dt, 0.0, 4.0, 30, 2, 1, 1, capi.GOFRT_SCREENED)
    s.reset(3)
    with pytest.raises(capi.AnlError, match="the cell changes along the trajectory"):
        s.calculate(0)
    ot, dt = _case(9, 768, 8, 12.0, None)
    g = capi.DeviceGofrt(dt, 0.0, 4.0, 30, 2)
    g.reset(3)
    ref, _ = O.gofrt(ot, 0.0, 4.0, 30, 2, 4, 1, 1, 3, 0, want_vdata=False)
    assert np.array_equal(g.calculate(0), ref) and g.stats()[0] == capi.GOFRT_FP64
