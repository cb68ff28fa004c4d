"""g(r,t) over the windows of a LAMMPS binary file, on a HIP runtime without
kernels: the order of each frame's atoms, which the screened form needs, is made
on the thread that reads the next window, while the current block computes, and
no position is read back from the device."""
import fake_hip

_SETUP = """
import os, tempfile
from analisi_amd import pyanalisi as pa
N, F, BLOCKS = 300, 61, 4
rng = np.random.default_rng(5)
L = 18.0
pos = rng.uniform(0, L, (F, N, 3))
box = np.tile(np.array([0, L, 0, L, 0, L], float), (F, 1))
types = (np.arange(N) % 2 + 1).astype(np.int32)
mem = pa.Trajectory(pos, np.zeros_like(pos), types, box, pa.BoxFormat.LammpsOrtho, False, False)
path = os.path.join(tempfile.mkdtemp(), "t.bin")
mem.write_lammps_binary(path, 0, -1)
me = None
def uploads(e, frames, threads):         # of an order of `frames` frames: 4 bytes an atom
    return [x for x in e if x[1] in ("memcpyasync", "memcpy") and x[2] == "1" and int(x[3]) == 4 * N * frames
            and (x[0] in threads)]
def read_back(e):
    return [x for x in e if x[1] == "memcpy" and x[2] == "2" and int(x[3]) % (32 * N) == 0]
"""


def test_block_average(tmp_path_factory):
    fake_hip.run(_SETUP + """
t = pa.Traj(path)
log()
pa.gofrt_block_average(t, BLOCKS, 0.0, 4.0, 16, 5, 1, 1)
e = log()
main = launches(e, "gofrt_screened_kernel")[0][0]
assert len(launches(e, "gofrt_screened_kernel")) == BLOCKS
assert not read_back(e), read_back(e)
window = {int(x[3]) // (4 * N) for x in e if x[1] == "memcpyasync" and x[2] == "1" and int(x[3]) % (4 * N) == 0
          and int(x[3]) // (4 * N) > 8}
others = {x[0] for x in e} - {main}
per_frames = [len(uploads(e, f, others)) for f in window]
assert max(per_frames) >= BLOCKS - 1, (window, per_frames)
# the calling thread makes the first window's only
assert all(len(uploads(e, f, {main})) <= 1 for f in window)
# and the others free nothing, which would wait for the running kernel
assert not [x for x in e if x[1] in ("free", "hostfree") and x[0] in others]
""", tmp_path_factory)


def test_in_memory_trajectory(tmp_path_factory):
    fake_hip.run(_SETUP + """
log()
g = pa.Gofrt(mem, 0.0, 4.0, 16, 5, 1, 1, 1, False)
g.reset(20)
g.calculate(0)
e = log()
assert launches(e, "gofrt_screened_kernel")
assert not read_back(e), read_back(e)
""", tmp_path_factory)


def test_only_for_the_objects_that_use_it(tmp_path_factory):
    """No order for an MSD's windows, nor for those of a plain FP64 g(r,t)."""
    fake_hip.run(_SETUP + """
t = pa.Traj(path)
log()
pa.msd_block_average(t, BLOCKS, 1, 5, False, False)
g = pa.Gofrt_lammps(t, 0.0, 4.0, 16, 5, 1, 1, 1, False, 0)
g.reset(8)
t.setAccessWindowSize(14)
for k in range(3):
    t.setAccessStart(14 * k)
    t.prefetch(14 * (k + 1))
    g.calculate(14 * k)
e = log()
assert launches(e, "gofrt_fp64_kernel") and launches(e, "msd_")
for frames in (14, 15, 16, 17, 18, 19, 20):
    assert not uploads(e, frames, {x[0] for x in e}), frames
assert not read_back(e)
""", tmp_path_factory)
