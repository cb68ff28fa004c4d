"""Which kernel and launch shape an MSD takes, on a HIP runtime without kernels
that refuses launches of 2^32 threads and more (the real one runs their number
modulo 2^32, without an error)."""
import fake_hip

_SETUP = """
import re
def trajectory(N, F, nt=1):
    box = np.tile(np.array([0, 0, 0, 5, 5, 5.0]), (F, 1))
    return capi.DeviceTrajectory(np.zeros((F, N, 3)), box, (np.arange(N) % nt).astype(np.int32), nt,
                                 np.zeros((F, nt, 3)))
def kernel(t, skip, tmax, n, cm_self=0):  # (R, W) of the window kernel, or "atoms"
    log()
    capi.msd(t, skip, tmax, 0, cm_self, n, 0)
    name = launches(log(), "msd_")[0][5]
    m = re.search(r"msd_window_kernelILi(\\d+)ELi(\\d+)E", name)
    return (int(m.group(1)), int(m.group(2))) if m else "atoms"
"""


def test_few_lags_per_residue(tmp_path_factory):
    """Strides near or above the number of lags: the window kernel while the chip
    is not full, eight lags per thread once it is."""
    fake_hip.run(_SETUP + """
t = trajectory(20000, 40)
assert kernel(t, 30, 16, 20) == (8, 4)               # a lag per residue, 313 x 16 workgroups
t = trajectory(50000, 90)
for tmax, n, cm, want in ((11, 66, 0, "atoms"), (33, 44, 0, "atoms"), (33, 55, 0, (8, 4)), (33, 55, 1, "atoms"),
                          (44, 46, 0, (8, 4))):      # 782 x 11 workgroups
    assert kernel(t, 11, tmax, n, cm) == want, (tmax, n, cm, kernel(t, 11, tmax, n, cm))
assert kernel(t, 1, 3, 2) != "atoms"
""", tmp_path_factory)


def test_chosen_shapes_at_strides(tmp_path_factory):
    """A chosen shape runs stride 1 always, other strides where a residue has a
    workgroup's lags; elsewhere the calculation's own does."""
    fake_hip.run(_SETUP + """
t = trajectory(640, 420)
own = {c: kernel(t, *c) for c in ((50, 200, 200), (3, 60, 200), (2, 200, 200), (1, 200, 200))}
for shape in t.MSD_SHAPES[:-1]:
    t.set_msd_tile(*shape)
    for c in own:
        lags = -(-c[1] // c[0])
        want = shape if c[0] == 1 or lags >= shape[0] * shape[1] else own[c]
        assert kernel(t, *c) == want, (shape, c, kernel(t, *c))
t.set_msd_tile(0)
assert all(kernel(t, *c) == "atoms" for c in own)
""", tmp_path_factory)


def test_many_blocks(tmp_path_factory):
    """More blocks than one launch can hold: launched in ranges."""
    fake_hip.run(_SETUP + """
t = trajectory(60, 12, nt=60)
nb, n = 290000, 4
for skip, name, most in ((1, "msd_window_kernel", 2), (4, "msd_atoms_kernel", 5)):
    log()
    b = capi.DeviceBlocks(t, [0] * nb, [n] * nb, msd=True, msd_skip=skip, msd_tmax=4, use_graph=False)
    b.run()
    e = log()
    fin, work = launches(e, "msd_finish_kernel"), launches(e, name)
    assert 1 < len(fin) <= most and len(work) == len(fin)
    assert all(int(x[3].split(",")[0]) * int(x[4]) < 2 ** 32 for x in fin + work)
    assert sum(int(x[3].split(",")[0]) for x in fin) >= nb * 60
    b.close()
""", tmp_path_factory)
