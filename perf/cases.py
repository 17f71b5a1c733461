"""The work that users of this package have it do, as measurable cases.

A simulation case is one sampling interval of a running production run: a
handle that has already left its random start advances `steps` Monte Carlo
steps and the observables of its state points are read back, as the drop-in
executable does for every row of data.out (and cluster.out) and as
scan_series does for every sample of a (T, P) scan.  The handle is what
such a program keeps; its launch plan is the default one, except where a
case says that the program autotuned it (then `plan` holds the tuning that
a cached autotune run applies).

A restart case loads a configuration into a handle, runs it on and reads
the whole lattice back, as a run with Flag_config = 1 does.  The reweighting
cases are the two halves of the histogram reweighting program: the Jacobi
sweeps of the constants, and the scan of (T, P) targets and angles.

Trajectories are fixed by the counter-based random numbers, so the
observables' integers are the same for every correct implementation; no
plain 64-bit formula gives them, and exact() has none for the simulation
cases.  The reweighting outputs have one.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cvfbulkwater_amd import (FP32_COMPENSATED, FP64, SCHED_FAST, SCHED_REFERENCE, VOLUME_DEVICE, VOLUME_HOST,
                              Params, Simulation)
from cvfbulkwater_amd.reweight import Reweighting

EQUILIBRATION = 64  # MC steps between the random start and the first measured interval


def listed():
    return [
        # the smallest production run: finite-size studies start at a few
        # hundred molecules; data.out row every 10 steps, latency is all
        {"name": "plain_L12", "kind": "plain", "L": 12, "T": 0.815, "P": 0.45, "steps": 10},
        # the reference's own production shape, the drop-in's default
        {"name": "plain_L32", "kind": "plain", "L": 32, "T": 0.815, "P": 0.45, "steps": 10},
        # Flag_chessboard = 0: eta fixed, hydrogen bonds gated by counters
        {"name": "nonchess_L32", "kind": "nonchess", "L": 32, "T": 0.815, "P": 0.45, "steps": 10},
        # Swendsen-Wang runs with data.out and cluster.out rows every 10
        # steps: the published isobar's size, and the large mixed-precision
        # lattice
        {"name": "cluster_L32", "kind": "cluster", "L": 32, "T": 0.70, "P": 0.45, "steps": 10, "n_cluster": 1,
         "fp32c": False},
        {"name": "cluster_L96", "kind": "cluster", "L": 96, "T": 0.65, "P": 0.30, "steps": 10, "n_cluster": 1,
         "fp32c": True},
        # a run restarted from input_config that ends with config.out
        {"name": "restart_L48", "kind": "restart", "L": 48, "T": 0.815, "P": 0.45, "steps": 64,
         "n_cluster": 0},
        # an isobar scan as isobar_scan runs it: one lattice size, a sample
        # of every point each 10 steps, no autotuning
        {"name": "scan_16x32", "kind": "scan", "points": 16, "sizes": "32", "steps": 10, "plan": "default",
         "fast": False},
        # the 128-point scan over four sizes, autotuned (the plan that the
        # autotuner picks), a sample after each 64-step sequence
        {"name": "batch_128", "kind": "scan", "points": 128, "sizes": "16,24,32,48", "steps": 64,
         "plan": "resident", "fast": False},
        # the same scan on the colour-pass schedule
        {"name": "fast_128", "kind": "scan", "points": 128, "sizes": "16,24,32,48", "steps": 64,
         "plan": "default", "fast": True},
        # one large lattice, beyond what one plane per CU holds
        {"name": "wide_L160", "kind": "wide", "L": 160, "T": 0.70, "P": 0.40, "steps": 10},
        # the reweighting constants at the program's production shape (11
        # simulations x 100,000 samples, BIN_FCT 2, STEP 300)
        {"name": "reweight_constants", "kind": "constants", "n_sim": 11, "samples": 100000, "bin_factor": 2.0,
         "sweeps": 300},
        # its scan: 64 (T, P) points x 3 mixing angles
        {"name": "reweight_scan", "kind": "rwscan", "n_sim": 11, "samples": 100000, "bin_factor": 2.0,
         "sweeps": 100, "targets": 64, "angles": 3},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _lattice(rng, lo, hi):
    """A lattice size: the chessboard needs a multiple of 4."""
    return min(max(4 * int(round(_log_int(rng, lo, hi) / 4)), lo), hi)


def draw(rng):
    kind = rng.choice(["plain", "plain", "nonchess", "cluster", "cluster", "restart", "scan", "scan", "wide",
                       "constants", "rwscan"])
    T, P = round(rng.uniform(0.55, 1.0), 4), round(rng.uniform(-0.1, 0.8), 4)
    if kind == "plain":
        return {"kind": kind, "L": _lattice(rng, 8, 64), "T": T, "P": P, "steps": rng.choice([1, 5, 10, 20, 33])}
    if kind == "nonchess":
        return {"kind": kind, "L": _lattice(rng, 8, 48), "T": T, "P": P, "steps": rng.choice([5, 10, 17])}
    if kind == "cluster":
        return {"kind": kind, "L": _lattice(rng, 8, 128), "T": T, "P": P, "steps": rng.choice([3, 5, 10]),
                "n_cluster": rng.choice([1, 1, 2]), "fp32c": rng.random() < 0.5}
    if kind == "restart":
        return {"kind": kind, "L": _lattice(rng, 8, 64), "T": T, "P": P, "steps": _log_int(rng, 10, 100),
                "n_cluster": rng.choice([0, 0, 1])}
    if kind == "scan":
        n = _log_int(rng, 3, 96)
        sizes = ",".join(str(_lattice(rng, 8, 48)) for _ in range(rng.choice([1, 1, 2, 3])))
        return {"kind": kind, "points": n, "sizes": sizes, "steps": rng.choice([5, 10, 25, 50]),
                "plan": rng.choice(["default", "default", "resident"]), "fast": rng.random() < 0.3}
    if kind == "wide":
        return {"kind": kind, "L": _lattice(rng, 100, 176), "T": T, "P": P, "steps": rng.choice([3, 5, 10])}
    case = {"kind": kind, "n_sim": rng.randint(2, 12), "samples": _log_int(rng, 3000, 90000),
            "bin_factor": rng.choice([0.5, 1.0, 2.0]), "sweeps": rng.randint(40, 250)}
    if kind == "rwscan":
        case |= {"targets": _log_int(rng, 5, 60), "angles": rng.randint(1, 4)}
    return case


# --------------------------------------------------------------- simulation
RESIDENT_PLAN = {"streams": 1, "fused": 2, "block_chunk": 1024, "graph_steps": 64}


def _points(case, seed):
    """State points of a case."""
    kind = case["kind"]
    if kind in ("plain", "restart"):
        return Params(L=case["L"], T=case["T"], P=case["P"], seed=seed, n_cluster=case.get("n_cluster", 0),
                      precision=FP64, volume_mode=VOLUME_HOST)
    if kind == "nonchess":
        return Params(L=case["L"], T=case["T"], P=case["P"], seed=seed, precision=FP64, volume_mode=VOLUME_HOST,
                      flag_chessboard=0)
    if kind == "cluster":
        return Params(L=case["L"], T=case["T"], P=case["P"], seed=seed, n_cluster=case["n_cluster"],
                      precision=FP32_COMPENSATED if case["fp32c"] else FP64,
                      volume_mode=VOLUME_DEVICE if case["fp32c"] else VOLUME_HOST)
    if kind == "wide":
        return Params(L=case["L"], T=case["T"], P=case["P"], seed=seed, precision=FP32_COMPENSATED,
                      volume_mode=VOLUME_DEVICE)
    # a (T, P) grid of eight temperatures; size i % n for point i
    sizes = [int(v) for v in case["sizes"].split(",")]
    return [Params(L=sizes[i % len(sizes)], T=0.55 + 0.45 * (i % 8) / 7, P=-0.10 + 0.06 * ((i // 8) % 16),
                   seed=seed + 1000003 * i, precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE,
                   schedule=SCHED_FAST if case["fast"] else SCHED_REFERENCE) for i in range(case["points"])]


def _rows(sim, n):
    """The observables of every state point, as a scan collects them."""
    real, whole = np.empty((n, 7)), np.empty((n, 3), np.int64)
    for i in range(n):
        o = sim.observe(i)
        real[i] = (o.E, o.H, o.V, o.n_hb, o.m, o.r_cell, o.E_vdw)
        whole[i] = (o.step, o.nhb2, o.n_sigma)
    return {"real": real, "whole": whole}


# -------------------------------------------------------------- reweighting
def _isobar(case, seed):
    """(h, rho) samples in internal units of an isobar crossing the critical
    region, each temperature a T-dependent mixture of a low- and a
    high-density phase; six digits, as the driver's awk prints them."""
    rng = np.random.default_rng(seed)
    n = case["samples"]
    T_hat = [0.1058 + 0.001 * k / max(case["n_sim"] - 1, 1) for k in range(case["n_sim"])]
    out = []
    for T in T_hat:
        hi = rng.random(n) < 1.0 / (1.0 + np.exp((T - 0.1063) / 0.0004))
        rho = np.where(hi, 0.690, 0.640) + 0.006 * rng.standard_normal(n)
        h = np.where(hi, -2.80, -2.72) + 0.012 * rng.standard_normal(n) + 0.5 * (rho - 0.665) + 0.8 * (T - 0.1063)
        out.append(np.stack([np.round(h, 5), np.round(rho, 6)], axis=1))
    return T_hat, [0.5] * len(T_hat), out


def _targets(case):
    """Scan targets (T K, P bar) and mixing angles."""
    n = case["targets"]
    T = np.array([(0.1060 + 0.0006 * k / max(n - 1, 1)) * 140.5678 + 185.4676 for k in range(n)])
    P = np.array([(0.5 + 0.0005 * (k % 4)) * 4694.59 - 2111.5552 for k in range(n)])
    return T, P, np.array([1.55 + 0.02 * a for a in range(case["angles"])])


RW_L = 8  # N = 512 molecules, the size of the critical-point study


# --------------------------------------------------------------- the cases
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("constants", "rwscan"):
        T_hat, P_hat, data = _isobar(case, seed)
        rw = Reweighting(RW_L, T_hat, P_hat, data, case["bin_factor"])
        state = {"kind": kind, "rw": rw, "sweeps": case["sweeps"]}
        if kind == "rwscan":
            rw.solve_constants(case["sweeps"])
            state["targets"] = _targets(case)
        return state
    pts = _points(case, seed)
    sim = Simulation(pts)
    n = 1 if isinstance(pts, Params) else len(pts)
    if case.get("plan") == "resident":
        sim.tuning = RESIDENT_PLAN
    sim.step(EQUILIBRATION)
    sim.sync()
    state = {"kind": kind, "sim": sim, "n": n, "steps": case["steps"]}
    if kind == "restart":
        state |= {"config": sim.get_config(), "labels": case["n_cluster"] > 0}
    return state


def run(state):
    kind = state["kind"]
    if kind == "constants":
        c, prev, converged = state["rw"].solve_constants(state["sweeps"])
        return {"c": c, "prev": prev, "converged": converged}
    if kind == "rwscan":
        T, P, alpha = state["targets"]
        return state["rw"].scan(T, P, alpha)
    sim = state["sim"]
    if kind == "restart":
        sigma, eta = state["config"]
        bad = sim.set_config(sigma, eta)
        sim.step(state["steps"])
        out = _rows(sim, 1)
        out["bad"] = bad
        out["sigma"], out["eta"] = sim.get_config()
        if state["labels"]:
            out["labels"] = sim.labels()
        return out
    sim.step(state["steps"])
    out = _rows(sim, state["n"])
    if kind == "cluster":
        c = sim.cluster_stats()
        out["cluster"] = np.array([c.largest, c.second, c.n_perc, c.n_clusters], np.int64)
        out["moments"] = np.array([c.mean, c.var], np.float32)
    return out


def _occupied(case):
    """Occupied cells of a reweighting case (a bound from its samples)."""
    return min(case["n_sim"] * case["samples"], 720_000)


def work(case):
    kind = case["kind"]
    if kind in ("constants", "rwscan"):
        # per sweep: every occupied cell's three doubles read once and, per
        # cell, an exponential per simulation and one per target (about 20
        # operations each)
        cells = _occupied(case)
        if kind == "constants":
            return {"bytes": 24.0 * cells * case["sweeps"],
                    "flops": 20.0 * cells * 2 * case["n_sim"] * case["sweeps"]}
        nt, na = case["targets"], case["angles"]
        # per target: log_P's exponential, the density's, and 10 operations
        # per angle; the densities are not an output
        return {"bytes": 28.0 * cells + 8.0 * 75 * nt * na,
                "flops": cells * (20.0 * case["n_sim"] + nt * (40.0 + 10.0 * na))}
    if kind == "scan":
        sizes = [int(v) for v in case["sizes"].split(",")]
        cells = sum(sizes[i % len(sizes)] ** 3 for i in range(case["points"]))
    else:
        cells = case["L"] ** 3
    # the 4-byte word of every cell read and written once per interval and
    # read once for the observables; per cell and step six sigma proposals
    # of about 35 integer operations each (a quarter of a Philox block among
    # them) and its share of a cube move
    nbytes, ops = 12.0 * cells, 230.0 * cells * case["steps"]
    if kind == "restart":
        nbytes += 24.0 * cells  # 12 bytes per cell in and out on the host side
    if case.get("n_cluster"):
        # Swendsen-Wang: five Philox blocks and 18 links per cell; the last
        # step's labels (six nodes per cell) written and read once
        nbytes += 48.0 * cells
        ops += 700.0 * cells * case["steps"] * case["n_cluster"]
    return {"bytes": nbytes, "flops": ops}


# ------------------------------------------------------------- 64-bit values
def _f32(x):
    return float(np.float32(x))


def _grid(case, seed):
    """Occupied cells of the (e, rho) histogram in simulation order, after
    histogram_reweighting_mixed_paramSI_norm_x.f90:81-283 (its conversion
    constants are single-precision literals)."""
    T_hat, P_hat, data = _isobar(case, seed)
    T = np.array(T_hat) * _f32(140.5678) + _f32(185.4676)
    P = np.array(P_hat) * _f32(4694.59) + _f32(-2111.5552)
    es, ds = [], []
    for t, p, s in zip(T_hat, P, data):
        d = _f32(1527.3) * s[:, 1] + _f32(-23.1017)
        es.append(_f32(11.272132) * s[:, 0] + _f32(9.028914) * t - _f32(1.8) * p / d)
        ds.append(d)
    e_all, d_all = np.concatenate(es), np.concatenate(ds)
    n_bin = int(np.sqrt(np.float32(case["samples"])) / np.float32(2))
    e_lo, e_range, d_lo, d_range = e_all.min(), np.ptp(e_all), d_all.min(), np.ptp(d_all)
    te, td = e_range / n_bin, d_range / n_bin
    n_bin += 20
    e_lo, e_range, d_lo, d_range = e_lo - 10 * te, e_range + 20 * te, d_lo - 10 * td, d_range + 20 * td
    nb = int(n_bin * 10 * case["bin_factor"])
    de, dd = e_range / nb, d_range / nb
    ids, weights = [], []
    for e, d in zip(es, ds):
        i, w = ((e - e_lo) / de).astype(np.int64), ((d - d_lo) / dd).astype(np.int64)
        ids.append(i * nb + w)
        weights.append(np.full(len(e), 1.0 / (len(e) * de * dd)))
    cell, where = np.unique(np.concatenate(ids), return_inverse=True)
    hist = np.bincount(where, np.concatenate(weights))
    e, d = e_lo + (cell // nb + 0.5) * de, d_lo + (cell % nb + 0.5) * dd
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    put = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=dev)  # noqa: E731
    N = RW_L ** 3
    return {"E": put(e * N), "V": put(_f32(0.018) / d * N), "lh": put(np.log(hist)), "e": put(e), "d": put(d),
            "area": de * dd, "nm": int(np.sqrt(np.float32(nb))), "beta": put(1000.0 / (_f32(0.2293) * T)),
            "p": put(P * 100.0), "lm": put(np.full(len(T), float(np.log(np.float32(case["samples"])))))}


def _terms(g, c):
    """The part of each simulation's argument that no target changes."""
    return -(g["beta"][:, None] * (g["E"] + g["p"][:, None] * g["V"])) - c[:, None] + g["lm"][:, None]


def _target(g, u, beta, p):
    """log_P of every cell at one target and log_Z (f90:1003-1124), with the
    program's two cut-offs of e^-10."""
    t1 = beta * (g["E"] + p * g["V"])
    top, low = u.max(0).values, u.min(0).values
    x = torch.exp(u - top)
    everything = torch.log(x.sum(0)) + top
    near = torch.log(torch.where(top - u < 10.0, x, torch.zeros_like(x)).sum(0)) + top
    cut = (t1 + top > 10.0) | (t1 + low < -10.0)
    lp = g["lh"] - (t1 + torch.where(cut, near, everything))
    m = lp.max()
    ex = torch.exp(lp - m)
    lz = torch.log(torch.where(m - lp < 10.0, ex, torch.zeros_like(ex)).sum()) + m
    return lp, lz


def _constants(g, sweeps):
    c = torch.zeros_like(g["beta"])
    prev = torch.zeros_like(c)
    for _ in range(sweeps):
        u = _terms(g, c)
        lz = torch.stack([_target(g, u, g["beta"][t], g["p"][t])[1] for t in range(len(c))])
        prev, c = c, lz - lz[0]
    return c, prev


def _moments(x, p, w):
    """norm 1, mean 0, variance 1 of a histogram p at x with bin widths w."""
    p = p / (p * w).sum()
    mean = (x * p * w).sum()
    x = x - mean
    norm, var = (p * w).sum(), (x * x * p * w).sum()
    a1 = math.sqrt(norm / var)
    return x * a1, p / (norm * a1), w * a1, mean, a1


def _order_parameter(g, v, alpha):
    """x, p, (mean, scale, Binder cumulant) of the mixed order parameter
    (f90:1383-1619, 2580-2608)."""
    nm = g["nm"]
    X = g["e"] * math.sin(alpha) + g["d"] * math.cos(alpha)
    lo, hi = float(X[v > 0].min()), float(X[v > 0].max())
    w = (hi - lo) / nm
    lo, w = lo - 2 * w, ((hi - lo) + 4 * w) / nm
    k = ((X - lo) / w).to(torch.int64)
    p = torch.zeros(nm, dtype=torch.float64, device=v.device).index_add_(0, k, v).cpu().numpy()
    x, p, wid, mean, _ = _moments(lo + (np.arange(nm) + 0.5) * w, p, np.full(nm, w))
    b, pi = _f32(1.53), _f32(3.14159)
    x = b * b * np.sin(pi * x / b) / (pi * pi) + x
    wid = np.concatenate([[x[1] - x[0]], (x[2:] - x[:-2]) / 2.0, [x[-1] - x[-2]]])
    x, p, wid, _, a1 = _moments(x, p, wid)
    m2 = (x / a1 + mean) ** 2
    q = p / p.sum()
    return x, p, (mean, a1, 1.0 - (m2 * m2 * q).sum() / (3.0 * (m2 * q).sum() ** 2))


def _ising3d(z):
    q = z * z / _f32(1.141059404) ** 2
    return _f32(0.436591191) * np.exp(-(q - 1) ** 2 * (_f32(0.196) * q + _f32(0.807)))


def _ising2d(z):
    return np.exp(-(_f32(0.058137) * z ** 16 + _f32(-2.68949) * z * z + _f32(-0.11235) * abs(z) + _f32(2.884162)))


def _scores(x, p):
    """Ising comparison of a distribution (f90:2042-2182)."""
    k = float(np.float32(6.0) / np.float32(0.8))
    z = np.linspace(0.1, 2.0, 2_000_001)
    on, out = p != 0, []
    f2, f3, q = _ising2d(x[on]), _ising3d(x[on]), p[on]
    out += [float(((np.log(f, where=f > 0, out=np.zeros_like(f)) - np.log(q)) * f).sum()) for f in (f2, f3)]
    out += [float((np.sqrt(q) * abs(q - f(x[on]))).sum() / ((f(z).max() - f(0.0)) * on.sum()))
            for f in (_ising2d, _ising3d)]
    mid = np.flatnonzero((x > -1) & (x < 1))
    i = mid[np.argmin(p[mid])]
    out.append((p[i] - _ising3d(0.0)) ** 2 * k * k + x[i] ** 2)
    height = 0.0
    for side, at in ((np.flatnonzero(x < 0), _f32(-1.14)), (np.flatnonzero(x >= 0), _f32(1.14))):
        i = side[np.argmax(p[side])]
        height += (p[i] - _ising3d(at)) ** 2 * k * k + (x[i] - at) ** 2
    return out + [height]


def exact(case, seed):
    if case["kind"] not in ("constants", "rwscan"):
        return None
    g = _grid(case, seed)
    c, prev = _constants(g, case["sweeps"])
    if case["kind"] == "constants":
        return {"c": c.cpu().numpy(), "prev": prev.cpu().numpy(), "converged": None}
    T, P, alpha = _targets(case)
    nt, na, nm = len(T), len(alpha), g["nm"]
    out = {"binder_ed": np.zeros((nt, 2)), "x": np.zeros((nt, na, nm)), "p": np.zeros((nt, na, nm)),
           "stats": np.zeros((nt, na, 3)), "scores": np.zeros((nt, na, 6))}
    u = _terms(g, c)
    for t in range(nt):
        lp, lz = _target(g, u, 1000.0 / (_f32(0.2293) * T[t]), P[t] * 100.0)
        v = torch.exp(lp - lz)
        v = v / (v.sum() * g["area"])
        for k, z in enumerate((g["e"], g["d"])):
            out["binder_ed"][t, k] = float(1.0 - ((v * z ** 4).sum() / v.sum()) /
                                           (3.0 * ((v * z ** 2).sum() / v.sum()) ** 2))
        for a in range(na):
            out["x"][t, a], out["p"][t, a], out["stats"][t, a] = _order_parameter(g, v, alpha[a])
            out["scores"][t, a] = _scores(out["x"][t, a], out["p"][t, a])
    return out
