"""Launches of the spherical densities and the order parameters on a HIP runtime
without kernels that refuses 2^32 threads and more (the real one runs their
number modulo 2^32, without an error)."""
import fake_hip


def test_many_frames(tmp_path_factory):
    """1,000 atoms x 68,000 frames within one density budget: 4.35e9 threads."""
    fake_hip.run("""
N, F = 1000, 68000
box = np.tile(np.array([0, 0, 0, 5, 5, 5.0]), (F, 1))
t = capi.DeviceTrajectory(np.zeros((F, N, 3)), box, np.zeros(N, np.int32), 1)
for sann in (False, True):
    h = capi.DeviceSph(t, [(0.5, 3.0)], 1, 2)
    if sann:
        h.set_neighbours([(8, 4.0, 4.0)])
    log()
    h.steinhardt(F, 1, 0, [2], 10, averaged=sann)
    e = log()
    d = launches(e, "sph_density")
    assert len(d) == 2
    for x in launches(e, "sph_"):
        assert int(x[3].split(",")[0]) * int(x[4]) < 2 ** 32
    threads = sum(int(x[3].split(",")[0]) * int(x[4]) for x in d)
    assert threads == 64 * N * F
    assert len({x[6:][-1] for x in d}) == 2
""", tmp_path_factory, timeout=300)
