"""The calculations whose speed is followed, as a user's program makes them.

A case is a dict of plain values; its "kind" names the operator:
  gofr  pyanalisi.Gofrt                     van Hove g(r,t) counts
  msd   pyanalisi.MeanSquareDisplacement
  gk    pyanalisi.GreenKubo                 FP64 lag correlations of one series
  gkb   capi.DeviceSeries.gk_blocks         all blocks of a block average in one call, FP64 or matrix cores
  sph   pyanalisi.SphericalCorrelations     lmax 10
  stein pyanalisi.SteinhardtOrderParameterHistogram_6

prepare() makes what a program holds before the call (a trajectory or a log and
the operator on it), run() is one reset / calculate / read of the result, and
exact() is the same result from plain numpy and torch in 64 bits.

Trajectories are a jittered lattice with shuffled types that then walks
randomly, unwrapped, at the atom densities of the test and benchmark
workloads; current series are AR(2) processes, as in analisi_amd.synth.
"""
import math

import numpy as np
import torch

from analisi_amd import capi, pyanalisi

LMAX_SPH = 10


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the reference test suite's g(r,t) call: a 56-atom solid cell, rmax over
        # half the shortest edge, 700 timesteps, every tenth one a time origin.
        # One of many such calls of a notebook: call overhead counts
        dict(name="gofr_test_cell", kind="gofr", N=56, density=0.268, types=3, F=712, n=700, tmax=10, skip=10, every=1,
             nbin=200, rmax=3.8, cell="ortho", sigma=0.05),
        # a small liquid, every timestep an origin, short lags (the smallest
        # benchmark workload)
        dict(name="gofr_small_liquid", kind="gofr", N=1000, density=0.03, types=2, F=201, n=150, tmax=51, skip=1,
             every=1, nbin=200, rmax=10.0, cell="cubic", sigma=0.05),
        # a constant-pressure run: the tilted cell is another one at every timestep
        dict(name="gofr_npt", kind="gofr", N=3000, density=0.09, types=2, F=120, n=100, tmax=20, skip=5, every=2,
             nbin=200, rmax=10.0, cell="npt", sigma=0.08),
        # the largest benchmark system, a window of 16 origins and 16 lags
        dict(name="gofr_large", kind="gofr", N=65536, density=0.0899, types=2, F=32, n=16, tmax=16, skip=1, every=1,
             nbin=512, rmax=15.0, cell="cubic", sigma=0.08),
        # the reference test suite's mean square displacement call
        dict(name="msd_test_cell", kind="msd", N=56, density=0.268, types=3, F=700, n=300, tmax=400, skip=10, cm=True,
             cm_self=False, cell="ortho", sigma=0.05),
        # diffusion of a liquid with drift removal, every timestep an origin
        # (the benchmark's lags on a smaller system)
        dict(name="msd_liquid", kind="msd", N=8192, density=0.09, types=2, F=1000, n=499, tmax=499, skip=1, cm=True,
             cm_self=True, cell="cubic", sigma=0.08),
        # the same with thinned time origins, as long runs are analysed; odd sizes
        dict(name="msd_thinned", kind="msd", N=4001, density=0.1, types=3, F=1500, n=1001, tmax=499, skip=10, cm=False,
             cm_self=False, cell="tri", sigma=0.08),
        # the reference test suite's Green-Kubo call on its 20,000-row log
        dict(name="gk_test_log", kind="gk", rows=20000, ncur=2, tmax=2000, n=18000, skip=1, n_seg=4, subtract=False,
             start_mean=0),
        # thermal conductivity of a two-component fluid from a long log
        dict(name="gk_long_log", kind="gk", rows=100001, ncur=2, tmax=5000, n=95001, skip=1, n_seg=1, subtract=True,
             start_mean=4000),
        # block average of a long log on the matrix cores
        dict(name="gk_blocks", kind="gkb", rows=500000, ncur=2, tmax=8000, n=23250, blocks=16, skip=1, n_seg=1,
             mfma=True),
        # density correlations of the local environment, four radial shells
        dict(name="sph_shells", kind="sph", N=512, density=0.05, types=2, F=300, n=150, tmax=150, skip=5, nbin=4,
             rmin=0.7, rmax=4.5, cell="cubic", sigma=0.03),
        # averaged order parameters over nearest-neighbour lists, q4 - q6 histogram
        dict(name="stein_averaged", kind="stein", N=2000, density=0.1, types=2, F=60, n=60, skip=2, nbin=1, rmin=0.5,
             rmax=3.0, hist=True, sann=True, averaged=True, cut=4.5, cap=80, cell="cubic", sigma=0.03),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: systems of tens to tens of thousands of
    atoms, logs of thousands to hundreds of thousands of rows, every cell and
    option, at most the listed ones' work."""
    kind = rng.choice(["gofr", "gofr", "gofr", "msd", "msd", "msd", "gk", "gk", "gkb", "sph", "stein"])
    if kind == "gofr":
        N = _log_int(rng, 40, 40000)
        cell = rng.choice(["cubic", "cubic", "tri", "tri", "npt"])
        tmax = _log_int(rng, 1, 60)
        n = _log_int(rng, 8, 700)
        skip = rng.choice([1, 1, 2, 5, 10])
        every = rng.choice([1, 1, 2, 3])
        # N^2 x origins x lags, and atoms x timesteps, within the listed ones
        lim = 2.5e10 if cell == "npt" else 8e11
        while N * N * (n / skip) * min(n, tmax) / every > lim or N * (n + tmax) > 2.5e6:
            if n > 16:
                n //= 2
            elif tmax > 1:
                tmax //= 2
            else:
                N //= 2
        rho = rng.uniform(0.03, 0.1)
        L = (N / rho) ** (1 / 3)
        return dict(kind="gofr", N=N, density=rho, types=rng.randint(1, 3), F=n + min(n, tmax) + rng.randint(0, 3), n=n,
                    tmax=tmax, skip=skip, every=every, nbin=rng.choice([50, 101, 200, 512]),
                    rmax=round(min(rng.uniform(4.0, 15.0), 0.44 * L), 3), cell=cell,
                    sigma=rng.choice([0.02, 0.05, 0.08]))
    if kind == "msd":
        N = _log_int(rng, 40, 30000)
        tmax = _log_int(rng, 8, 800)
        n = _log_int(rng, 50, 2000)
        skip = rng.choice([1, 1, 2, 5, 10, 17])
        while N * (n + tmax) > 1.2e7 or N * (n / skip) * min(n, tmax) > 2e9:
            n = max(20, n // 2)
            tmax = max(8, tmax // 2)
            N = max(40, int(N / 1.5))
        return dict(kind="msd", N=N, density=rng.uniform(0.03, 0.1), types=rng.randint(1, 3),
                    F=n + min(n, tmax) + rng.randint(0, 3), n=n, tmax=tmax, skip=skip, cm=rng.random() < 0.5,
                    cm_self=rng.random() < 0.5, cell=rng.choice(["cubic", "tri"]), sigma=rng.choice([0.02, 0.05, 0.08]))
    if kind == "gk":
        tmax = _log_int(rng, 100, 6000)
        n = _log_int(rng, max(500, tmax), 95000)
        skip = rng.choice([1, 1, 1, 2, 5])
        return dict(kind="gk", rows=n + tmax + rng.randint(0, 50), ncur=rng.randint(1, 3), tmax=tmax, n=n, skip=skip,
                    n_seg=rng.choice([1, 1, 4]), subtract=rng.random() < 0.3, start_mean=tmax * 3 // 4)
    if kind == "gkb":
        tmax = _log_int(rng, 200, 8000)
        blocks = rng.randint(2, 16)
        n = _log_int(rng, tmax, max(tmax + 1, 360000 // blocks))
        return dict(kind="gkb", rows=blocks * n + tmax + rng.randint(0, 50), ncur=rng.randint(1, 2), tmax=tmax, n=n,
                    blocks=blocks, skip=1, n_seg=1, mfma=rng.random() < 0.5)
    N = _log_int(rng, 60, 2000)
    cell = rng.choice(["cubic", "cubic", "tri"])
    if kind == "sph":
        tmax = _log_int(rng, 10, 150)
        n = _log_int(rng, tmax, 300)
        while N * (n + tmax) > 1.2e5:
            N = max(60, N // 2)
            n = max(tmax, n // 2)
            if N == 60:
                break
        rho = rng.uniform(0.04, 0.08)
        L = (N / rho) ** (1 / 3)
        return dict(kind="sph", N=N, density=rho, types=rng.randint(1, 2), F=n + tmax + rng.randint(0, 3), n=n,
                    tmax=tmax, skip=rng.choice([1, 5, 10]), nbin=rng.choice([1, 3, 4]), rmin=0.5,
                    rmax=round(min(rng.uniform(3.0, 5.0), 0.44 * L), 3), cell=cell, sigma=0.03)
    n = _log_int(rng, 10, 100)
    while N * n > 1.2e5:
        n //= 2
    rho = rng.uniform(0.04, 0.1)
    L = (N / rho) ** (1 / 3)
    sann = rng.random() < 0.6
    return dict(kind="stein", N=N, density=rho, types=rng.randint(1, 2), F=n, n=n, skip=rng.choice([1, 2, 3]),
                nbin=1 if sann else rng.choice([1, 3]), rmin=0.5, rmax=round(min(3.5, 0.44 * L), 3),
                hist=rng.random() < 0.6, sann=sann, averaged=sann and rng.random() < 0.5,
                cut=round(min(4.5, 0.44 * L), 3), cap=100, cell=cell, sigma=0.03)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _trajectory(c, seed):
    """(positions [F][N][3], types [N], boxes [F][6 or 9] in the LAMMPS order)"""
    rng = np.random.default_rng([seed, 17])
    N, F = c["N"], c["F"]
    L = (N / c["density"]) ** (1.0 / 3.0)
    if c["cell"] == "ortho":  # edges in the proportions 4.14 : 7.82 : 6.45
        e = np.array([4.14141307, 7.81544411, 6.44646321])
        edge = e * (L / np.prod(e) ** (1.0 / 3.0))
    else:
        edge = np.array([L, L, L])
    k = np.maximum(1, np.ceil(N ** (1.0 / 3.0) * edge / L)).astype(int)
    while np.prod(k) < N:
        k[np.argmin(k / edge)] += 1
    site = rng.permutation(int(np.prod(k)))[:N]
    frac = np.stack(np.unravel_index(site, tuple(k)), axis=1) + rng.uniform(0.2, 0.8, (N, 3))
    frac = frac / k
    tilt = np.array([0.11, -0.08, 0.06]) * L if c["cell"] in ("tri", "npt") else None
    x0 = frac * edge
    if tilt is not None:
        x0[:, 0] += frac[:, 1] * tilt[0] + frac[:, 2] * tilt[1]
        x0[:, 1] += frac[:, 2] * tilt[2]
    pos = rng.standard_normal((F, N, 3))
    pos *= c["sigma"]
    pos[0] = x0
    np.cumsum(pos, axis=0, out=pos)
    box = np.zeros((F, 6 if tilt is None else 9))
    box[:, [1, 3, 5]] = edge
    if tilt is not None:
        box[:, 6:] = tilt
    if c["cell"] == "npt":  # edges and tilts breathe by about half a per cent, the atoms with them
        s = 1.0 + 0.005 * np.sin(0.3 * np.arange(F))[:, None] + 0.001 * rng.standard_normal((F, 1))
        box[:, [1, 3, 5]] *= s
        box[:, 6:] *= s
        pos *= s[:, :, None]
    types = rng.permutation(N).astype(np.int32) % max(1, c["types"])
    return pos, np.sort(types), box


def _currents(c, seed):
    """[rows][3 ncur] of AR(2) currents, each after the first correlated with it"""
    rng = np.random.default_rng([seed, 23])
    T, nc = c["rows"], c["ncur"]
    # x_t = 1.6 x_{t-1} - 0.7 x_{t-2} + e_t through its impulse response, which
    # falls below 1e-16 within 400 terms
    h = np.zeros(512)
    h[0], h[1] = 1.0, 1.6
    for i in range(2, 512):
        h[i] = 1.6 * h[i - 1] - 0.7 * h[i - 2]
    nf = 1 << (T + 511).bit_length()
    e = rng.standard_normal((3 * nc, T))
    x = np.fft.irfft(np.fft.rfft(e, nf) * np.fft.rfft(h, nf), nf)[:, :T]
    for k in range(1, nc):
        x[3 * k:3 * k + 3] = 0.3 * x[:3] + math.sqrt(1 - 0.09) * x[3 * k:3 * k + 3]
    return np.ascontiguousarray(x.T)


def _headers(nc):
    return ["j%d[%d]" % (k, i + 1) for k in range(nc) for i in range(3)]


def _lists(c):
    return [(c["cap"], c["cut"] ** 2, c["cut"] ** 2)] * c["types"] if c.get("sann") else []


def prepare(c, seed):
    kind = c["kind"]
    if kind in ("gk", "gkb"):
        data = _currents(c, seed)
        if kind == "gkb":
            return dict(case=c, series=capi.DeviceSeries(data), primo=[b * c["n"] for b in range(c["blocks"])],
                        n=[c["n"]] * c["blocks"], idx=[3 * k for k in range(c["ncur"])])
        names = _headers(c["ncur"])
        log = pyanalisi.ReadLog(data, names)
        op = pyanalisi.GreenKubo(log, "", c["skip"], names[::3], False, c["tmax"], 2, c["subtract"], c["start_mean"],
                                 c["n_seg"], False, 1, 100)
        return dict(case=c, data=data, log=log, op=op)
    pos, types, box = _trajectory(c, seed)
    fmt = pyanalisi.BoxFormat.LammpsTriclinic if box.shape[1] == 9 else pyanalisi.BoxFormat.LammpsOrtho
    traj = pyanalisi.Trajectory(pos, np.zeros_like(pos), types, box, fmt, False, False)
    if kind == "gofr":
        op = pyanalisi.Gofrt(traj, 0.0, c["rmax"], c["nbin"], c["tmax"], 1, c["skip"], c["every"], False)
    elif kind == "msd":
        op = pyanalisi.MeanSquareDisplacement(traj, c["skip"], c["tmax"], 1, c["cm"], c["cm_self"], False)
    else:
        ranges = [(c["rmin"], c["rmax"])] * c["types"] ** 2
        if kind == "sph":
            op = pyanalisi.SphericalCorrelations(traj, ranges, c["nbin"], c["tmax"], 1, c["skip"], 10, False, [])
        else:
            op = pyanalisi.SteinhardtOrderParameterHistogram_6(traj, ranges, c["nbin"], 100, [4, 6], 1, c["skip"],
                                                               c["hist"], _lists(c), c["averaged"])
    return dict(case=c, traj=traj, op=op)


def run(state):
    c = state["case"]
    if c["kind"] == "gkb":
        per, mean, var = state["series"].gk_blocks(state["idx"], c["skip"], c["tmax"], c["n_seg"], False, 0,
                                                   state["primo"], state["n"], mfma=c["mfma"])
        return [per, mean, var]
    op = state["op"]
    op.reset(c["n"])
    op.calculate(0)
    return np.array(op, copy=True)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(c):
    kind = c["kind"]
    if kind in ("gk", "gkb"):
        nb = c.get("blocks", 1)
        leff = min(c["n"], c["tmax"])
        n0 = -(-c["n"] // c["skip"])
        narr = 3 * c["ncur"] ** 2 + 2
        return dict(bytes=8.0 * (nb * c["n"] + leff) * 3 * c["ncur"] + 8.0 * nb * leff * narr,
                    flops=6.0 * c["ncur"] ** 2 * nb * n0 * leff)
    N, nt = c["N"], c["types"]
    n0 = -(-c["n"] // c["skip"])
    if kind == "stein":
        nb = _neighbours(c)
        frames = c["n"] // c["skip"]
        out = c["nbin"] * nt * nt * 1e4 if c["hist"] else c["nbin"] * frames * N * nt * 6.0
        # each pair's distance once per direction, 49 harmonics of each neighbour
        return dict(bytes=24.0 * frames * N + 8 * out, flops=frames * N * nb * (10.0 + 4 * 49))
    leff = min(c["n"], c["tmax"])
    frames = min(c["F"], c["n"] + leff)
    read = 24.0 * N * frames
    if kind == "msd":
        return dict(bytes=read + 8.0 * leff * nt * 2, flops=9.0 * N * n0 * leff)
    if kind == "sph":
        dens = 121.0 * nt * c["nbin"] * N
        return dict(bytes=read + 8.0 * leff * nt * nt * c["nbin"] * 11,
                    flops=2.0 * dens * n0 * leff + frames * N * _neighbours(c) * (10.0 + 4 * 121))
    # g(r,t): the distances of the pairs that are counted (10 operations and a bin each)
    lags = -(-leff // c["every"])
    return dict(bytes=read + 8.0 * leff * nt * (nt + 1) * c["nbin"], flops=12.0 * N * _neighbours(c) * n0 * lags)


def _neighbours(c):
    r = c["cut"] if c.get("sann") else c["rmax"]
    return min(c["N"], 1.0 + c["density"] * 4.19 * r ** 3)


# ---------------------------------------------------------------------------
# the results in plain 64-bit arithmetic
# ---------------------------------------------------------------------------
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _image(d, b):
    """minimum image of the vectors d (last axis) in the cell b (LAMMPS order): z, then y, then x"""
    L = [b[1] - b[0], b[3] - b[2], b[5] - b[4]]
    x, y, z = d[..., 0], d[..., 1], d[..., 2]
    k = torch.round(z / L[2])
    z = z - k * L[2]
    if len(b) == 9:
        y = y - k * b[8]
        x = x - k * b[7]
    k = torch.round(y / L[1])
    y = y - k * L[1]
    if len(b) == 9:
        x = x - k * b[6]
    x = x - torch.round(x / L[0]) * L[0]
    return x, y, z


def _exact_gofr(c, pos, types, box):
    N, nt, nbin = c["N"], c["types"], c["nbin"]
    leff = min(c["n"], c["tmax"])
    t0s, lags = range(0, c["n"], c["skip"]), range(0, leff, c["every"])
    if N * N * len(t0s) * len(lags) > 6e9 or len(t0s) * len(lags) > 9000:
        return None
    dev = _dev()
    P = torch.tensor(pos, device=dev)
    ty = torch.tensor(types, device=dev, dtype=torch.int64)
    half = nt * (nt + 1) // 2
    a, b = torch.minimum(ty[:, None], ty[None]), torch.maximum(ty[:, None], ty[None])
    ch = half - torch.div((b + 1) * (b + 2), 2, rounding_mode="floor") + a
    ch = ch + half * torch.eye(N, device=dev, dtype=torch.int64)
    dr = c["rmax"] / nbin
    out = torch.zeros((leff, 2 * half * nbin), device=dev, dtype=torch.float64)
    for lag in lags:
        for t0 in t0s:
            x, y, z = _image(P[t0][:, None] - P[t0 + lag][None], box[t0])
            r = torch.sqrt(x * x + y * y + z * z)
            u = torch.floor((r / dr).float()).to(torch.int64)
            ok = (r <= c["rmax"]) & (u < nbin)
            out[lag] += torch.bincount((ch * nbin + u)[ok], minlength=2 * half * nbin)
    incr = 1.0 / int(c["n"] // c["skip"]) if c["n"] >= c["skip"] else 1.0
    return (out * incr).reshape(leff, 2 * half, nbin).cpu().numpy()


def _exact_msd(c, pos, types):
    nt = c["types"]
    leff = min(c["n"], c["tmax"])
    dev = _dev()
    P = torch.tensor(pos, device=dev)
    ty = torch.tensor(types, device=dev, dtype=torch.int64)
    cm = torch.stack([P[:, ty == t].mean(1) for t in range(nt)], 1)
    Q = P - cm[:, ty] if c["cm_self"] else P
    out = np.zeros((leff, 2 if c["cm"] else 1, nt))
    for lag in range(leff):
        e = ((Q[0:c["n"]:c["skip"]] - Q[lag:lag + c["n"]:c["skip"]]) ** 2).sum(2).mean(0)
        for t in range(nt):
            out[lag, 0, t] = float(e[ty == t].mean())
        if c["cm"]:
            out[lag, 1] = ((cm[0:c["n"]:c["skip"]] - cm[lag:lag + c["n"]:c["skip"]]) ** 2).sum(2).mean(0).cpu().numpy()
    return out


def _gk_block(J, c, n, leff):
    """[leff][3 ncur^2 + 2] of the block that starts at row 0 of J"""
    nc = c["ncur"]
    seg = n // c["n_seg"]
    nf = 1 << (n + leff).bit_length()
    dev = _dev()
    X = torch.tensor(J[:n + leff].T.copy(), device=dev)
    FB = torch.fft.rfft(X, nf)
    C = torch.zeros((nc, nc, leff), device=dev, dtype=torch.float64)
    for s in range(c["n_seg"]):
        first = seg * s + (seg * s) % c["skip"]
        m = torch.zeros(n + leff, device=dev, dtype=torch.float64)
        m[first:seg * (s + 1):c["skip"]] = 1.0
        FA = torch.fft.rfft(X * m, nf)
        for a in range(nc):
            for b in range(nc):
                p = (FA[3 * a:3 * a + 3].conj() * FB[3 * b:3 * b + 3]).sum(0)
                C[a, b] += torch.fft.irfft(p, nf)[:leff] / float(m.sum()) / 3.0 / c["n_seg"]
    C = C.reshape(nc * nc, leff).cpu().numpy()
    if c.get("subtract") and c["start_mean"] < leff:
        C = C - C[:, c["start_mean"]:].mean(1, keepdims=True)
    out = np.zeros((leff, 3 * nc * nc + 2))
    out[:, :nc * nc] = C.T
    it = np.arange(1, leff)
    integral = np.cumsum(C[:, :-1] / 2 + C[:, 1:] / 2, axis=1)
    einst = np.cumsum(C[:, :-1] * it / 2 + C[:, 1:] * it / 2, axis=1) / it
    out[1:, nc * nc:3 * nc * nc:2] = integral.T
    out[1:, nc * nc + 1:3 * nc * nc:2] = einst.T
    for col, M in ((0, integral), (1, integral - einst)):
        M = M.T.reshape(leff - 1, nc, nc)
        M = (M + M.transpose(0, 2, 1)) / 2
        with np.errstate(all="ignore"):
            if nc == 1:
                k = M[:, 0, 0]
            elif nc == 2:
                k = M[:, 0, 0] - M[:, 0, 1] * (1.0 / M[:, 1, 1]) * M[:, 1, 0]
            else:
                k = np.full(leff - 1, np.nan)
                ok = np.abs(M[:, 1:, 1:]).max((1, 2)) > 0
                k[ok] = M[ok, 0, 0] - np.einsum("ki,kij,kj->k", M[ok, 0, 1:], np.linalg.inv(M[ok, 1:, 1:]),
                                                M[ok, 1:, 0])
        out[1:, 3 * nc * nc + col] = k
    return out


def _harmonics(x, y, z, lmax):
    """real orthonormal harmonics up to a sign per (l, m): [(lmax+1)^2][...], block l at l^2"""
    r = torch.sqrt(x * x + y * y + z * z)
    ct = z / r
    st = torch.sqrt(x * x + y * y) / r
    ph = torch.atan2(y, x)
    Y = [None] * (lmax + 1) ** 2
    pmm = torch.ones_like(r)
    for m in range(lmax + 1):
        if m:
            pmm = pmm * st * (2 * m - 1)
        p1, p2 = pmm, torch.zeros_like(r)
        for l in range(m, lmax + 1):
            p = p1 if l == m else (ct * (2 * l - 1) * p1 - (l + m - 1) * p2) / (l - m)
            if l > m:
                p1, p2 = p, p1
            k = math.sqrt((2 * l + 1) / (4 * math.pi) * math.factorial(l - m) / math.factorial(l + m))
            if m == 0:
                Y[l * l + l] = k * p
            else:
                Y[l * l + l + m] = math.sqrt(2) * k * p * torch.cos(m * ph)
                Y[l * l + l - m] = math.sqrt(2) * k * p * torch.sin(m * ph)
    return torch.stack(Y)


def _sann(d, cut, ty, nt):
    """chosen [N][N]: the nearest-neighbour rule on the distances d, per neighbour type"""
    N = d.shape[0]
    chosen = torch.zeros_like(d, dtype=torch.bool)
    for t in range(nt):
        w = torch.where((ty[None] == t) & (d <= cut), d, torch.full_like(d, math.inf))
        r, order = torch.sort(w, dim=1)
        n = torch.isfinite(r).sum(1)
        s = torch.cumsum(torch.where(torch.isfinite(r), r, torch.zeros_like(r)), 1)
        m = torch.arange(N, device=d.device)
        # stops at the first m >= 3 with sum of the first m distances <= r_m (m - 2), or at the list's end
        stop = torch.zeros_like(chosen)
        stop[:, 3:] = s[:, 2:-1] <= r[:, 3:] * (m[3:] - 2.0)
        stop |= m[None] >= n[:, None]
        stop[:, :3] = False
        k = torch.where(n >= 3, torch.where(stop.any(1), stop.to(torch.int8).argmax(1), n), torch.zeros_like(n))
        chosen |= torch.zeros_like(chosen).scatter(1, order, m[None] < k[:, None])
    return chosen


def _densities(c, x, types, b, lmax):
    """S [N][nt][nbin][(lmax+1)^2], neighbour counts [N][nt][nbin] and, with lists, the chosen pairs of one frame"""
    nt, nbin, N = c["types"], c["nbin"], c["N"]
    dx, dy, dz = _image(x[:, None] - x[None], b)
    r = torch.sqrt(dx * dx + dy * dy + dz * dz)
    r.fill_diagonal_(math.inf)
    if c.get("sann"):
        ok = _sann(r, c["cut"], types, nt)
        u = torch.zeros_like(types[:, None] + types[None])
    else:
        dr = (c["rmax"] - c["rmin"]) / nbin
        u = torch.floor(((r - c["rmin"]) / dr).float())
        ok = (u >= 0) & (u < nbin)
        u = torch.where(ok, u, torch.zeros_like(u)).to(torch.int64)
    i, j = torch.nonzero(ok, as_tuple=True)
    Y = _harmonics(dx[i, j], dy[i, j], dz[i, j], lmax)
    at = (i * nt + types[j]) * nbin + u[i, j]
    S = torch.zeros((N * nt * nbin, Y.shape[0]), device=x.device, dtype=torch.float64)
    S.index_add_(0, at, Y.T.contiguous())
    n = torch.bincount(at, minlength=N * nt * nbin)
    return S.reshape(N, nt, nbin, -1), n.reshape(N, nt, nbin).double(), ok if c.get("sann") else None


def _exact_sph(c, pos, types, box):
    leff = min(c["n"], c["tmax"])
    if c["N"] ** 2 * (c["n"] + leff) > 1.5e9:
        return None
    dev = _dev()
    ty = torch.tensor(types, device=dev, dtype=torch.int64)
    P = torch.tensor(pos, device=dev)
    nt, L1 = c["types"], LMAX_SPH + 1
    S = torch.stack([_densities(c, P[t], ty, box[t], LMAX_SPH)[0] for t in range(c["n"] + leff - 1)])
    out = np.zeros((leff, nt, nt, c["nbin"], L1))
    for lag in range(leff):
        p = (S[0:c["n"]:c["skip"]] * S[lag:lag + c["n"]:c["skip"]]).mean(0)
        for l in range(L1):
            q = p[..., l * l:(l + 1) ** 2].sum(-1)
            for t in range(nt):
                out[lag, t, :, :, LMAX_SPH - l] = q[ty == t].mean(0).cpu().numpy()
    return out


def _exact_stein(c, pos, types, box):
    nt, nbin, N, lmax = c["types"], c["nbin"], c["N"], 6
    if N ** 2 * c["n"] > 1.5e9:
        return None
    frames = c["n"] // c["skip"]
    dev = _dev()
    ty = torch.tensor(types, device=dev, dtype=torch.int64)
    q = np.zeros((nbin, frames, N, nt, lmax))
    hist = np.zeros((nbin, nt, nt, 100 * 100))
    for f in range(frames):
        t = f * c["skip"]
        S, n, ok = _densities(c, torch.tensor(pos[t], device=dev), ty, box[t], lmax)
        m = S
        if c["averaged"]:
            w = S / n[..., None]
            m = torch.zeros_like(S)
            for jt in range(nt):
                a = (ok & (ty[None] == jt)).double()
                near = w[:, jt, 0].clone()
                # a neighbour without neighbours of this type makes the sum undefined
                bad = torch.isnan(near).any(1)
                near[bad] = 0.0
                v = a @ near
                v = torch.where(((a @ bad.double()) > 0)[:, None], torch.full_like(v, math.nan), v)
                own = torch.where((ty == jt)[:, None], S[:, jt, 0] / n[:, jt, 0][:, None], torch.zeros_like(v))
                m[:, jt, 0] = own + v
        v = torch.stack([(m[..., l * l:(l + 1) ** 2] ** 2).sum(-1) * 4 * math.pi / (2 * l + 1)
                         for l in range(1, lmax + 1)], -1)
        v = torch.sqrt(v / n[..., None] / n[..., None])
        v = torch.where((n > 0)[..., None], v, torch.zeros_like(v))
        q[:, f] = v.permute(2, 0, 1, 3).cpu().numpy()
        if c["hist"]:
            cell = torch.floor((v * 100).float())
            cell = torch.where(cell < 100, cell, torch.full_like(cell, 99)).to(torch.int64)
            h = cell[..., 3] * 100 + cell[..., 5]
            for it in range(nt):
                for jt in range(nt):
                    for b in range(nbin):
                        use = (ty == it) & (n[:, jt, b] > 0)
                        hist[b, it, jt] += torch.bincount(h[use, jt, b], minlength=10000).cpu().numpy()
    return (hist / frames).reshape(nbin, nt, nt, 100, 100) if c["hist"] else q


def exact(c, seed):
    kind = c["kind"]
    if kind in ("gk", "gkb"):
        J = _currents(c, seed)
        leff = min(c["n"], c["tmax"])
        if kind == "gk":
            return _gk_block(J, c, c["n"], leff)
        per = np.stack([_gk_block(J[b * c["n"]:], c, c["n"], leff) for b in range(c["blocks"])])
        with np.errstate(invalid="ignore"):
            return [per, per.mean(0), per.var(0, ddof=1) / c["blocks"]]
    pos, types, box = _trajectory(c, seed)
    if kind == "gofr":
        return _exact_gofr(c, pos, types, box)
    if kind == "msd":
        return _exact_msd(c, pos, types)
    return _exact_sph(c, pos, types, box) if kind == "sph" else _exact_stein(c, pos, types, box)
