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


def test_many_blocks(tmp_path_factory):
    """More blocks than one launch can hold: launched in ranges."""
    fake_hip.run(_SETUP + """
t = trajectory(60, 12, nt=60)
nb, n = 290000, 4
for skip in (1, 4):
    log()
    b = capi.DeviceBlocks(t, [0] * nb, [n] * nb, msd=True, msd_skip=skip, msd_tmax=4, use_graph=False)
    b.run()
    e = log()
    fin, work = launches(e, "msd_finish_kernel"), launches(e, "msd_window_kernel")
    assert len(fin) == len(work) == 2
    assert all(int(x[3].split(",")[0]) * int(x[4]) < 2 ** 32 for x in fin + work)
    assert sum(int(x[3].split(",")[0]) for x in fin) >= nb * 60
    b.close()
""", tmp_path_factory)
