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


_SMALL = """
def system(N, F=30, nt=1, nbin=1, lmax=2):
    box = np.tile(np.array([0, 0, 0, 5, 5, 5.0]), (F, 1))
    t = capi.DeviceTrajectory(np.zeros((F, N, 3)), box, (np.arange(N) % nt).astype(np.int32), nt)
    h = capi.DeviceSph(t, [(0.5, 3.0)] * nt ** 2, nbin, lmax)
    h.set_neighbours([(8, 4.0, 4.0)] * nt)
    log()
    return h
"""


def test_averaged_form_fills_the_chip(tmp_path_factory):
    """Items per workgroup of the averaged order parameter: 64 for a large
    calculation, fewer where that leaves less than 2,048 workgroups."""
    fake_hip.run(_SMALL + """
for N, F, nt, nbin, want in ((10, 1, 1, 1, 3), (200, 20, 1, 1, 1000), (300, 20, 3, 6, 2077), (2000, 30, 2, 1, 2143),
                             (20000, 20, 1, 1, 6250)):
    h = system(N, F, nt, nbin)
    h.steinhardt(F, 1, 0, [2], 4, averaged=True)
    x = launches(log(), "sph_steinhardt_kernel")
    assert len(x) == 1 and int(x[0][3].split(",")[0]) == want, (N, x[0][3])
""", tmp_path_factory)


def test_small_calls_launch_no_more_than_they_need(tmp_path_factory):
    """The densities' Gram values are reduced and laid out by one kernel, once a
    chunk; neighbour lists of few atoms take no bounding spheres."""
    fake_hip.run(_SMALL + """
def names(e):
    return [x[5].split("sph_")[1].split("_kernel")[0] for x in launches(e, "sph_")]
h = system(100, 40)
h.calculate(20, 10, 2, 0)
assert names(log()) == ["zero", "density_sann", "gram_mfma", "reduce"]
h = system(640, 40)
h.calculate(20, 10, 2, 0)
assert names(log()) == ["zero", "density_sann", "gram_mfma", "reduce"]
h = system(1024, 8)                                   # few frames of more atoms
h.calculate(4, 4, 1, 0)
assert names(log()) == ["zero", "density_sann", "gram_mfma", "reduce"]
h = system(641, 40)
h.calculate(20, 10, 2, 0)
assert names(log()) == ["zero", "block_radius", "density_sann", "gram_mfma", "reduce"]
h.set_budget(5 * 641 * 9 * 8)                         # densities of two t1 values and their lags
h.calculate(4, 4, 1, 0)
n = names(log())
assert n.count("reduce") == n.count("gram_mfma") == 2 and n[-1] == "reduce", n
""", tmp_path_factory)
