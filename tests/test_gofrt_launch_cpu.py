"""g(r,t) launches on a HIP runtime without kernels that refuses 2^32 threads and
more (the real one runs their number modulo 2^32, without an error): longer
calculations go in ranges that cover every lag and t0 once."""
import fake_hip


def test_ranges(tmp_path_factory):
    fake_hip.run("""
import struct
N, F = 10, 8400
box = np.tile(np.array([0, 0, 0, 5, 5, 5.0]), (F, 1))
varying = box + np.arange(F)[:, None] * 1e-6 * np.array([0, 0, 0, 1, 1, 1.0])
def fields(e):                           # of GofrtArgs: k0, k1, chunk; first lag, lags, work items
    raw = bytes.fromhex(e[-1][1:])
    i = raw.find(struct.pack("<QII", 0, 4200, 0)) + 16
    assert i >= 16
    k = struct.unpack_from("<III", raw, i)
    j = raw.find(struct.pack("<ii", -2 ** 31, 2 ** 31 - 1)) + 8
    lag0, ntiles, nlag, nwork = struct.unpack_from("<4I", raw, j)
    return k, lag0, nlag, nwork
for b, form in ((box, 2), (box, 0), (varying, 2)):
    t = capi.DeviceTrajectory(np.zeros((F, N, 3)), b, np.zeros(N, np.int32), 1)
    for tune in ((4, 0), (8, 1)):
        g = capi.DeviceGofrt(t, 0.0, 3.0, 4, 4200, 1, 1, form)
        g.set_tuning(*tune, 1, 0)
        g.reset(4200)
        fake.fake_dump(512)
        log()
        g.calculate(0)
        e = launches(log(), "gofrt_")
        assert len(e) >= 2
        seen = np.zeros((4200, 4200), np.uint8)
        for x in e:
            assert int(x[3].split(",")[0]) * int(x[4]) < 2 ** 32
            (k0, k1, chunk), lag0, nlag, nwork = fields(x)
            seen[lag0:lag0 + nlag, k0:min(k1, k0 + nwork * chunk)] += 1
        assert (seen == 1).all()
""", tmp_path_factory)


def test_short_work_shares_workgroups(tmp_path_factory):
    """A workgroup whose t0 are short work takes several, as its start and the
    reading of its counters cost more than they do; one whose t0 are long work
    takes one where that fills the chip."""
    fake_hip.run("""
def workgroups(N, n, lags, rel, form, vary=False, bins=100):
    F = n + lags
    box = np.tile(np.array([0, 0, 0, 5, 5, 5.0]), (F, 1))
    if vary: box += np.arange(F)[:, None] * 1e-6 * np.array([0, 0, 0, 1, 1, 1.0])
    t = capi.DeviceTrajectory(np.zeros((F, N, 3)), box, np.zeros(N, np.int32), 1)
    g = capi.DeviceGofrt(t, 0.0, rel * 10, bins, lags, 1, 1, form)
    g.reset(n)
    log()
    g.calculate(0)
    e = launches(log(), "gofrt_")
    return sum(int(x[3].split(",")[0]) for x in e)
assert 512 <= workgroups(30, 200, 100, 0.3, 2) <= 1200
assert 100 <= workgroups(30, 200, 100, 0.3, 0) <= 1300
assert 512 <= workgroups(300, 100, 50, 0.3, 2) <= 3000
assert 1600 <= workgroups(4000, 40, 10, 0.1, 2) <= 3200
assert 512 <= workgroups(1000, 150, 40, 0.3, 0, True) <= 24000
assert workgroups(8000, 12, 6, 0.3, 2) == 32 * 6 * 12      # one t0 each
assert workgroups(8000, 12, 6, 0.3, 2, True) == 32 * 6 * 12
assert workgroups(2000, 3, 2, 0.3, 2) == 8 * 2 * 3         # fewer than fill the chip
""", tmp_path_factory)
