"""The plain FP64 g(r,t) against the oracle, counts bit-exact, on both sides of
its two launch shapes (a t0 per pair of wavefronts with 64 i, or 256 i per
workgroup) and around their tiles: one atom to several tiles, cells whose
minimum image needs one step, several or none, pairs at bin edges, cutoffs
beyond half of the cell, atom ranges and blocks."""
import numpy as np
import pytest

from analisi_amd import capi, synth
from gpu_util import first_diff
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _case(seed, N, F, L, tilt, shift=0.0):
    box = synth.lammps_box(L, tilt)
    pos = synth.random_walk(seed, N, F, box, 0.2)
    if shift:
        pos[:, ::3] += shift
        pos[:, 1::4] -= 1.7 * shift
    ot = O.Traj(pos, synth.types_by_fraction(N, [0.5, 0.3, 0.2]), np.tile(box, (F, 1)), tilt is not None)
    return ot, capi.DeviceTrajectory(ot.pos, ot.box, ot.type_id, ot.ntypes, ot.cm)


@pytest.mark.parametrize("N", [3, 31, 32, 33, 63, 64, 65, 97, 767, 768, 769, 1025])
@pytest.mark.parametrize("tilt,shift", [(None, 0.0), (None, 53.0), ([2.0, -1.6, 1.2], 0.0), ([-1.9, 1.4, 1.8], -47.0)])
def test_counts(N, tilt, shift):
    ot, dt = _case(3, N, 14, 8.0, tilt, shift)
    for rmin, rmax, nbin, skip, every, n, primo in [(0.0, 6.5, 200, 1, 1, 9, 0), (0.7, 4.5, 1, 3, 2, 8, 2)]:
        ref, _ = O.gofrt(ot, rmin, rmax, nbin, 4, 8, skip, every, n, primo, want_vdata=False)
        g = capi.DeviceGofrt(dt, rmin, rmax, nbin, 4, skip, every, capi.GOFRT_FP64)
        g.reset(n)
        got = g.calculate(primo)
        assert first_diff(got, ref) is None, first_diff(got, ref)
        st = g.pair_stats()
        assert g.stats()[0] == capi.GOFRT_FP64 and st["fp64"] == st["all"] == N * N * -(-n // skip) * -(-4 // every)


@pytest.mark.parametrize("N", [60, 800])
@pytest.mark.parametrize("rmin", [0.0, 0.2])
def test_pairs_at_bin_edges(N, rmin):
    """Pairs within ulps of every bin edge, of rmin and of rmax, coinciding
    atoms and an atom with itself at lag 0."""
    rmax, nbin = 5.0, 20
    rng = np.random.default_rng(4)
    box = np.tile(synth.lammps_box(9.0), (3, 1))
    pos = rng.uniform(0, 9, (3, N, 3))
    for k in range(N // 2):
        d = rmin + (k % (nbin + 1)) * ((rmax - rmin) / nbin)
        d = np.nextafter(d, [-np.inf, np.inf][k % 2]) if k % 3 else d
        pos[:, 2 * k + 1] = pos[:, 2 * k]
        pos[:, 2 * k + 1, k % 3] += d
    ot = O.Traj(pos, np.zeros(N, np.int32), box, False)
    dt = capi.DeviceTrajectory(ot.pos, ot.box, ot.type_id, ot.ntypes, ot.cm)
    ref, _ = O.gofrt(ot, rmin, rmax, nbin, 2, 4, 1, 1, 2, 0, want_vdata=False)
    g = capi.DeviceGofrt(dt, rmin, rmax, nbin, 2, form=capi.GOFRT_FP64)
    g.reset(2)
    got = g.calculate(0)
    assert first_diff(got, ref) is None, first_diff(got, ref)


@pytest.mark.parametrize("N", [100, 900])
def test_atom_ranges_and_blocks(N):
    ot, dt = _case(7, N, 30, 9.0, [1.0, 0.8, -0.7])
    g = capi.DeviceGofrt(dt, 0.2, 6.0, 33, 6, form=capi.GOFRT_FP64)
    g.reset(9)
    for t, im, a0, a1 in [(0, 0, 0, N), (3, 5, 17, 18), (5, 2, 40, N - 9), (1, 8, N - 1, N), (2, 1, 50, 50)]:
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
