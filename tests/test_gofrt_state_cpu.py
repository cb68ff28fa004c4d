"""State that g(r,t) calculations of one trajectory share, on a HIP runtime
without kernels: what a failed call leaves behind, and what each launch is
given while other calculations run."""
import fake_hip

_SETUP = """
rng = np.random.default_rng(3)
def trajectory(N=500, F=12, L=20.0, varying=False):
    pos = rng.uniform(0, L, (F, N, 3))
    box = np.zeros((F, 9))
    box[:, 3:6] = L / 2
    if varying:
        box[:, 3] += 0.01 * np.arange(F)
    return capi.DeviceTrajectory(pos, box[:, :6].copy(), np.zeros(N, np.int32), 1)
def words(entry):
    return {x.split(":")[0] for x in entry[6:]}
"""


def test_fractions_after_a_failed_allocation(tmp_path_factory):
    """Each of the allocations of the screen's fractions refused once: the call
    fails, frees what it had, and the next one builds all of them."""
    fake_hip.run(_SETUP + """
def new():
    t = trajectory()
    g = capi.DeviceGofrt(t, 0.0, 4.0, 20, 4)
    g.reset(6)
    return t, g
t, g = new()
log()
g.calculate(0)
e = log()
want = words(launches(e, "gofrt_screened_kernel")[0])
assert len(want) >= 8
refused = 0
for after in range(8):
    t, g = new()
    live = fake.fake_live()
    fake.fake_refuse(NEVER, after)
    try:
        g.calculate(0)
        ok = True
    except capi.AnlError as err:
        ok = False
    fake.fake_refuse(NEVER, NEVER)
    if ok:
        break
    refused += 1
    log()
    left = fake.fake_live()
    g.calculate(0)
    got = launches(log(), "gofrt_screened_kernel")[0]
    assert words(got) == want, (after, sorted(got[6:]))
    assert left <= live + (after > 0)                 # at most the pooled workspace
assert refused >= 4
""", tmp_path_factory)


def test_two_cutoffs_at_once(tmp_path_factory):
    """A calculation that another handle of the trajectory, with another rmax,
    runs in the middle of is launched with its own screen."""
    fake_hip.run(_SETUP + """
t = trajectory()
a, b = [capi.DeviceGofrt(t, 0.0, r, 20, 4) for r in (7.0, 2.0)]
a.reset(6)
b.reset(6)
a.calculate(0)
b.calculate(0)
def values(entries):                     # of the launch, without its addresses
    e = launches(entries, "gofrt_screened_kernel")
    assert len(e) == 1
    raw = bytes.fromhex(e[0][-1][1:])
    ptr = {int(x.split(":")[0]) for x in e[0][6:-1]}
    return [raw[8 * k:8 * k + 8] for k in range(len(raw) // 8) if k not in ptr]
fake.fake_dump(480)
log()
a.calculate(0)
alone = values(log())
seen = []
def other():
    if not seen:
        seen.append(log())
        b.calculate(0)
        seen.append(values(log()))
cb = WAIT(other)
fake.fake_wait(0, ctypes.cast(cb, ctypes.c_void_p))
a.calculate(0)
fake.fake_wait(0, None)
e = log()
assert len(seen) == 2 and not launches(seen[0], "gofrt_screened_kernel")
assert seen[1] != alone
assert values(e) == alone
""", tmp_path_factory)


def test_shape_from_the_environment(tmp_path_factory):
    """Each of the environment's launch settings, like anl_gofrt_set_tuning, is a
    choice of the shape: the default cluster mode is then kept where an untuned
    calculation would leave it (here groups 12 A wide in a cell of 40)."""
    fake_hip.run(_SETUP + """
import os
fake.fake_fill(0x41)                      # 0x41414141: a radius of 12.1 A
t = trajectory(L=40.0)
def kernel(env, tune=None):
    os.environ.update(env)
    g = capi.DeviceGofrt(t, 0.0, 4.0, 20, 4)
    for k in env:
        del os.environ[k]
    if tune:
        g.set_tuning(*tune)
    g.reset(6)
    log()
    g.calculate(0)
    return launches(log(), "gofrt_screened_kernel")[0][5]
untuned = kernel({})
chosen = kernel({}, (4, 1, 1 << 26, 2))
assert untuned != chosen
for env in (dict(ANL_GOFRT_UNROLL="4"), dict(ANL_GOFRT_XCD="1"), dict(ANL_GOFRT_PAIRS_PER_WG=str(1 << 26)),
            dict(ANL_GOFRT_CLUSTER="2")):
    assert kernel(env) == chosen, env
""", tmp_path_factory)
