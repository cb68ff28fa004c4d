"""The segment means of the FP64 Green-Kubo form (n_seg > 1) on a HIP runtime
without kernels: which memory each launch is given.  Calls that run at once do
not share it, a stream waits for the call that used it before, a captured
launch holds no address of it, and a call that cannot have it does without."""
import fake_hip

SEGM = 11  # the word of GkArgs that holds the segment means

_SETUP = """
def seg_of(entries):
    l = launches(entries, "gk_chain_kernel") + launches(entries, "gk_dense_kernel")
    return [dict(x.split(":") for x in e[6:]).get("%d") for e in l]
import ctypes
J = np.zeros((9000, 6))
s = capi.DeviceSeries(J)
idx = np.array([0, 3], np.uint32)
def run_async(out, tmax, n, stream=None):
    p, k = np.zeros(1, np.uint64), np.full(1, n, np.uint32)
    capi.check(capi.lib().anl_gk_calculate_blocks_async(s.handle, capi._ptr(idx), 2, 1, tmax, 4, 0, 0, capi._ptr(p),
               capi._ptr(k), 1, capi.GK_FP64, out, None, None, stream))
def device(nbytes):
    p = ctypes.c_void_p()
    assert fake.hipMalloc(ctypes.byref(p), ctypes.c_size_t(nbytes)) == 0
    return p
log()
""" % SEGM


def test_synchronous_calls_that_overlap(tmp_path_factory):
    """A second, larger call made while the first has not ended: memory of its
    own, and the first one's is not freed."""
    fake_hip.run(_SETUP + """
for blocks in (False, True):
    inner = []
    outer = []
    def other():
        outer.extend(log() if not inner else [])
        if not inner and launches(outer, "gk_"):
            s.gk([0, 3], 1, 3000, 5000, 4, False, 0, 0) if not blocks else s.gk_blocks(
                [0, 3], 1, 2000, 4, False, 0, [0, 100], [4000, 4000])
            inner.extend(log())
    cb = WAIT(other)
    fake.fake_wait(0, ctypes.cast(cb, ctypes.c_void_p))
    s.gk([0, 3], 1, 500, 3000, 4, False, 0, 0) if not blocks else s.gk_blocks(
        [0, 3], 1, 300, 4, False, 0, [0, 100], [2000, 2000])
    fake.fake_wait(0, None)
    a, b = seg_of(outer), seg_of(inner)
    assert len(a) == 1 and len(b) == 1 and a[0] and b[0], (a, b)
    assert a[0] != b[0]
    first = [e[6:] for e in launches(outer, "gk_chain")]
    held = {x.split(":")[1] for l in first for x in l}
    assert not [e for e in inner if e[1] == "free" and e[2] in held]
""", tmp_path_factory)


def test_asynchronous_calls_on_two_streams(tmp_path_factory):
    fake_hip.run(_SETUP + """
st = [ctypes.c_void_p(0xa0), ctypes.c_void_p(0xb0)]
out = device(3000 * 14 * 8)
run_async(out, 3000, 5000, st[0])
run_async(out, 400, 900, st[1])
e = log()
assert len(set(seg_of(e))) == 1 and seg_of(e)[0]      # the same memory,
last = max(i for i, x in enumerate(e) if x[1] == "launch" and x[2] == "0xa0")
first = min(i for i, x in enumerate(e) if x[1] == "launch" and x[2] == "0xb0")
rec = [x for x in e[last:first] if x[1] == "record" and x[3] == "0xa0"]
wait = [x for x in e[last:first] if x[1] == "waitevent" and x[2] == "0xb0"]
assert rec and wait and rec[-1][2] == wait[-1][3]     # after the first call's end
""", tmp_path_factory)


def test_captured_call_keeps_no_address(tmp_path_factory):
    fake_hip.run(_SETUP + """
s.gk([0, 3], 1, 3000, 5000, 4, False, 0, 0)
out = device(3000 * 14 * 8)
run_async(out, 3000, 5000)
log()
fake.fake_capture(1)
run_async(out, 400, 900)
fake.fake_capture(0)
e = log()
assert seg_of(e) == [None] * 4 and not launches(e, "gk_segments_kernel"), e
assert not [x for x in e if x[1] in ("malloc", "free", "record", "waitevent")]
""", tmp_path_factory)


def test_no_memory_for_the_segments(tmp_path_factory):
    """A device with room for the outputs only."""
    fake_hip.run(_SETUP + """
seg = 3000 * 14 * 8 + 256                 # more than the output
out = device(3000 * 14 * 8)
fake.fake_refuse(seg, NEVER)
r = s.gk([0, 3], 1, 3000, 5000, 4, False, 0, 0)
e = log()
assert seg_of(e) == [None] * 4 and not launches(e, "gk_segments_kernel")
run_async(out, 3000, 5000)
e = log()
assert seg_of(e) == [None] * 4
r = s.gk_blocks([0, 3], 1, 300, 4, False, 0, [0, 100, 200], [2000, 2000, 2000])
e = log()
assert len(seg_of(e)) == 1 and seg_of(e)[0]           # these fit
fake.fake_refuse(NEVER, NEVER)
r = s.gk([0, 3], 1, 3000, 5000, 4, False, 0, 0)
assert seg_of(log())[0]
""", tmp_path_factory)


def test_matrix_form_from_two_threads(tmp_path_factory):
    """The MFMA form's scratch: what one call enqueues on it is not mixed with
    another thread's."""
    fake_hip.run(_SETUP + """
import threading
fake.fake_launch_time(2000)
go = threading.Barrier(2)
def work(tmax):
    go.wait()
    for _ in range(5):
        s.gk([0, 3], 1, tmax, 2000, 2, False, 0, 0, mfma=True)
ts = [threading.Thread(target=work, args=(t,)) for t in (300, 500)]
[t.start() for t in ts]
[t.join() for t in ts]
e = launches(log(), "gkm_")
runs = [e[0][0]]
for x in e:
    if x[0] != runs[-1]:
        runs.append(x[0])
per_call = len(e) // 10
assert per_call >= 4 and len(runs) <= 10, (per_call, len(runs))
at = 0
while at < len(e):                        # whole calls, one after the other
    assert len({x[0] for x in e[at:at + per_call]}) == 1
    at += per_call
""", tmp_path_factory)


def test_copy_threads_sleep_while_the_kernels_run(tmp_path_factory):
    """gk_blocks' copy threads: a device that takes two seconds keeps less
    than half a core of the host busy (eight when the threads look all the time;
    the kernel counts their time in ticks, which is coarse)."""
    fake_hip.run(_SETUP + """
import resource, time
def cpu():
    r = resource.getrusage(resource.RUSAGE_SELF)
    return r.ru_utime + r.ru_stime
primo = list(range(0, 1400, 50))
used = []
for wait in (0, 0, 1000000):
    fake.fake_wait(wait, None)
    c, t = cpu(), time.perf_counter()
    s.gk_blocks([0, 3], 500, 1000, 1, False, 0, primo, [2000] * len(primo), stats=False)  # 3 MB, two pieces
    used.append(cpu() - c)
    t = time.perf_counter() - t
assert t > 1.9 and used[2] < t / 2, (used, t)
""", tmp_path_factory)


def test_few_terms_a_lag(tmp_path_factory):
    """Lags of few t0 take one launch of a thread each, however many segments and
    whether or not their means could be kept; longer ones do not."""
    fake_hip.run(_SETUP + """
def names(f):
    log()
    f()
    return [x[5].split("gk_")[1].split("_kernel")[0] for x in launches(log(), "gk_")][:-2]  # without the epilogue
gk = lambda n, tmax, skip, g: names(lambda: s.gk([0, 3], skip, tmax, n, g, False, 0, 0))
assert gk(2, 2, 1, 1) == ["few"]
assert gk(31, 30, 1, 100) == gk(53, 53, 65, 2) == gk(50, 50, 1, 4000000) == ["few"]
assert gk(3000, 2000, 1000, 30) == ["few"]
assert gk(200, 100, 1, 1) == ["chain"]
assert gk(4000, 2000, 1, 4) == ["chain", "segments"]
fake.fake_capture(1)
out = device(2000 * 14 * 8)
assert names(lambda: run_async(out, 2000, 4000)) == ["chain"] * 4
assert names(lambda: run_async(out, 10, 20)) == ["few"]
fake.fake_capture(0)
assert [len(gk(4500, 4000, 4294967280, 1)), len(gk(4500, 4500, 1, 1))] == [1, 1]
""", tmp_path_factory)
