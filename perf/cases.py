"""The framework's workloads as timed cases: what a program that uses it has it do, through
its public entry points, from one sweep of a few wavefronts to launches that fill the GPU.

A case is a dict of plain values.  ``prepare`` makes what a program holds before the call
(parameter sets, plans, networks, device buffers), ``run`` is one call and returns its
outputs whole, ``work`` counts the bytes and operations the call cannot do without and
``exact`` gives the outputs in 64 bits where they are computed numbers (the Monte Carlo's
counts are whole numbers of a fixed random stream and have no such value).

Kinds
  sweep   Context.run_fixed_dt into host arrays: the launch behind simulate()
  decay   a prepared plan of one isothermal set, launched into device buffers
  uneven  a persistent, graph-captured plan of many uneven parameter sets
  large   a prepared plan of clusters beyond one workgroup's LDS
  event   mcl_run_event into device buffers: the reference's loop, one event per step
  lab     Context.run_lab: TL_lab experiments with dose filling
  curves  CurveKind.mc_curves: Monte Carlo curves of a population of parameter sets
  glow    Context.glow_curve_device: binning and smoothing of per-step counts
  infer   Network.forward: surrogate curves of a batch
  train   train(): AdamW steps of the surrogate network, and its parameters afterwards
  search  NetworkDE: the network-scored differential evolution of a fit
"""
from __future__ import annotations

import ctypes as C
import math
from pathlib import Path

import numpy as np
import torch

from mcluminescence_amd import autotune, fit
from mcluminescence_amd import surrogate as S
from mcluminescence_amd import workloads as W
from mcluminescence_amd._abi import (DEFAULT_SEED, F_DEVICE_PTRS, F_GRAPH, F_PERSISTENT, Context,
                                     RunParams, Stats, run_array)

WEIGHTS = Path(S.__file__).with_name("surrogate_tl.npz")
LAYERS = (S.N_IN, 512, 512, 512, 512, S.N_BINS)          # the surrogate network's widths
# TL_lab rows: heating to the listed temperature over the duration under dose, from empty
LAB_ROWS = ((1086.0, 275.0), (2171.55, 250.0), (3257.33, 225.0), (4343.0, 200.0), (5429.0, 175.0),
            (6514.66, 150.0), (7600.0, 125.0), (8686.0, 100.0), (9772.0, 75.0), (10858.0, 50.0),
            (11944.0, 25.0))


def listed():
    return [
        # simulate() on the 16 x 500 thermoluminescence glow: a handful of clusters, where the
        # chain of steps and the host round trip are all there is
        {"name": "glow_16x500", "kind": "sweep", "physics": "trap", "electrons": 500, "sims": 16,
         "rate": 1.0, "steps": 4000, "bins": 0},
        # the isothermal decay ensemble of the benchmark: one launch that fills the GPU
        {"name": "decay_4096x400", "kind": "decay", "electrons": 400, "sims": 4096, "T": 500.0,
         "steps": 4000},
        # a sweep of uneven sets (64-2048 electrons, half ramps, half isothermal), 256-bin curves
        {"name": "sweep_10000", "kind": "uneven", "sets": 10000, "steps": 1024, "bins": 256},
        # large clusters, whose holes exceed a workgroup's LDS
        {"name": "large_250x8000", "kind": "large", "electrons": 8000, "sims": 250, "rate": 1.0,
         "steps": 4000},
        # the reference's own loop (rows of lum, time and electron ratio) on its TL12 physics
        {"name": "event_4096x400", "kind": "event", "electrons": 400, "sims": 4096, "rate": 5.0,
         "rows": 1280},
        # the objective of the lab fit with many simulations a row
        {"name": "lab_11x4096", "kind": "lab", "rows": 11, "sims": 4096, "sets": 1, "fill": False},
        # training and validation curves of the isothermal surrogate
        {"name": "curves_iso_64", "kind": "curves", "curve": "iso", "sets": 64, "sims": 32,
         "electrons": 400},
        # plotting's glow curves of a large sweep
        {"name": "glow_curves_1024", "kind": "glow", "runs": 1024, "sims": 16, "steps": 4000,
         "rate": 1.0, "width": 1.0},
        # surrogate curves of one odd-sized population: latency and launches
        {"name": "infer_300", "kind": "infer", "batch": 300},
        # surrogate curves of a large batch: throughput
        {"name": "infer_65536", "kind": "infer", "batch": 65536},
        # an epoch of surrogate training
        {"name": "train_b4096", "kind": "train", "rows": 65536, "batch": 4096},
        # the search of a surrogate-assisted fit
        {"name": "search_1024", "kind": "search", "pop": 1024, "gens": 150},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sweep", "sweep", "decay", "uneven", "large", "event", "lab", "curves",
                       "glow", "infer", "infer", "train", "search"])
    if kind == "sweep":
        return {"kind": kind, "physics": rng.choice(["trap", "tunnelling", "two_channel", "iso"]),
                "electrons": _log(rng, 50, 2000), "sims": _log(rng, 1, 64),
                "rate": rng.choice([0.5, 1.0, 2.0, 5.0]), "steps": rng.randint(700, 4000),
                "bins": rng.choice([0, 0, 256])}
    if kind == "decay":
        return {"kind": kind, "electrons": _log(rng, 50, 1500), "sims": _log(rng, 100, 4096),
                "T": round(rng.uniform(460.0, 560.0), 1), "steps": rng.randint(1000, 4000)}
    if kind == "uneven":
        return {"kind": kind, "sets": _log(rng, 300, 9999), "steps": rng.choice([512, 777, 1024]),
                "bins": rng.choice([64, 200, 256])}
    if kind == "large":
        return {"kind": kind, "electrons": rng.randint(3600, 7900), "sims": _log(rng, 8, 240),
                "rate": rng.choice([1.0, 2.0]), "steps": rng.randint(2000, 4000)}
    if kind == "event":
        rate = rng.choice([2.0, 5.0, 10.0])
        n = _log(rng, 30, 600)
        return {"kind": kind, "electrons": n, "sims": _log(rng, 16, 3000), "rate": rate,
                "rows": 900 + n}
    if kind == "lab":
        return {"kind": kind, "rows": rng.randint(1, 11), "sims": _log(rng, 1, 1000),
                "sets": rng.choice([1, 1, 15, 40]), "fill": rng.choice([False, True])}
    if kind == "curves":
        return {"kind": kind, "curve": rng.choice(["tl", "iso"]), "sets": _log(rng, 1, 64),
                "sims": rng.randint(4, 64), "electrons": rng.randint(200, 1000)}
    if kind == "glow":
        return {"kind": kind, "runs": _log(rng, 1, 1000), "sims": rng.randint(1, 16),
                "steps": rng.randint(500, 4000), "rate": rng.choice([0.5, 1.0, 5.0]),
                "width": rng.choice([0.5, 1.0, 2.0])}
    if kind == "infer":
        return {"kind": kind, "batch": _log(rng, 1, 65000)}
    if kind == "train":
        batch = 64 * _log(rng, 4, 128)
        return {"kind": kind, "rows": batch * rng.randint(4, 12) + rng.randint(0, 63), "batch": batch}
    return {"kind": kind, "pop": _log(rng, 64, 4000), "gens": rng.choice([25, 50, 100])}


# ---------------------------------------------------------------- inputs ------------------
_CTX = None


def _ctx():
    """The program's context, made once."""
    global _CTX
    if _CTX is None:
        _CTX = Context(0)
    return _CTX


def _runs(c):
    """Parameter sets of a sweep, decay, large or event case."""
    n, sims = c["electrons"], c["sims"]
    if c["kind"] == "decay":
        r = W.iso_decay_4096x400(sims=sims)[0]
        r.N_e = r.holes = float(n)
        r.T_start, r.n_steps = c["T"] - 273.15, c["steps"]
        return [r]
    if c["kind"] == "event":
        return W.tunnelling_tl12(sims=sims, n=n, T_rate=c["rate"])     # dt: a 1 K step cap below
    steps, rate = c["steps"], c["rate"]
    physics = c.get("physics", "trap")
    if physics == "trap":                     # 300 -> 700 K
        return [W.single_trap(1.3, 1e12, 4e9, 1e23, n, T_start_K=300.0, T_rate=rate,
                              dt=400.0 / rate / steps, n_steps=steps, sims=sims)]
    if physics == "iso":
        return W.tunnelling_iso(1e-4, n=n, fill=0.5, dt=1.0, n_steps=steps, sims=sims)
    r = W.tunnelling_tl12(sims=sims, n=n, T_rate=rate)[0]
    r.n_steps = steps
    r.dt = 800.0 / rate / steps
    if physics == "two_channel":
        r.E_loc_1, r.E_loc_2, r.Retrap = 1.15, 1.25, 0.3
    return [r]


def _params(seed):
    """Weights and biases of a fresh network, flat."""
    rng = np.random.default_rng(seed)
    parts = []
    for k, n in zip(LAYERS[:-1], LAYERS[1:]):
        lim = 1.0 / math.sqrt(k)
        parts += [rng.uniform(-lim, lim, n * k), rng.uniform(-lim, lim, n)]
    return np.concatenate(parts).astype(np.float32)


def _inputs(n, seed):
    """Encoded parameter sets, uniform in the box."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand((n, S.N_IN), generator=g, device="cuda") * 2.0 - 1.0


def _targets(x):
    """Smooth log-normalised peaks whose place, width and height follow the parameters."""
    t = torch.linspace(0.0, 1.0, S.N_BINS, device=x.device)
    mid = 0.5 + 0.3 * x[:, :1]
    width = 0.08 + 0.04 * x[:, 1:2]
    height = 0.02 * (1.2 + x[:, 4:5])
    c = height * torch.exp(-0.5 * ((t - mid) / width) ** 2) * (1.0 + 0.2 * x[:, 5:6] * (t - mid))
    return (torch.log1p(c.clamp_min(0.0) / S.C0) / math.log1p(1.0 / S.C0)).contiguous()


def _glow_counts(c, seed):
    """Per-step counts around a glow peak at 490 K on a 300 -> 700 K ramp."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    steps = c["steps"]
    T = 300.0 + 400.0 * torch.arange(steps, device="cuda") / steps
    mean = 500.0 * (400.0 / steps) * torch.exp(-0.5 * ((T - 490.0) / 18.0) ** 2) / 45.0
    lam = mean.expand(c["runs"] * c["sims"], steps)
    return torch.poisson(lam, generator=g).to(torch.int32).contiguous()


def _glow_runs(c):
    return [RunParams.make(T_start=26.85, T_rate=c["rate"], dt=400.0 / c["rate"] / c["steps"],
                           n_steps=c["steps"], sims=c["sims"]) for _ in range(c["runs"])]


def _lab_runs(c):
    runs, obs = [], []
    for k in range(c["sets"]):
        for duration, T_end in LAB_ROWS[:c["rows"]]:
            runs.append(RunParams.make(
                alpha=9e9, b=1e12, s=1e13, E_cb=1.8, E_loc_1=1.4 + 0.002 * k, E_loc_2=1.4 + 0.002 * k,
                D0=400.35, Retrap=0.5, k_b=W.K_B, D=0.092, rho_prime=1e-4, holes=100.0,
                boundary_factor=1.2, N_e=100.0, e_ratio_start=0.0, T_start=300.0,
                T_rate=(T_end - 300.0) / duration, dt=1.0, n_steps=1, sims=c["sims"]))
            obs.append([duration])
    return runs, obs


def prepare(case, seed):
    c = dict(case)
    kind, key = c["kind"], DEFAULT_SEED + seed
    st = {"case": c, "kind": kind, "seed": key}
    if kind == "sweep":
        st["runs"] = run_array(_runs(c))
    elif kind in ("decay", "large", "uneven"):
        runs = W.uneven_sweep(c["sets"], seed=seed, n_steps=c["steps"]) if kind == "uneven" else _runs(c)
        ctx = st["ctx"] = Context(0)
        if kind != "large":
            autotune.apply(ctx, runs)
        flags = F_PERSISTENT | F_GRAPH if kind == "uneven" else 0
        plan = st["plan"] = ctx.plan(runs, seed=key, n_bins=c.get("bins", 0), flags=flags)
        n, row = plan.info.total_clusters, plan.info.row_len
        st["counts"] = torch.zeros((n, row), dtype=torch.int32, device="cuda")
        st["live"] = torch.zeros(n, dtype=torch.int64, device="cuda")
    elif kind == "event":
        runs = _runs(c)
        runs[0].dt = 1.0
        st["runs"], n, rows = run_array(runs), c["sims"], c["rows"]
        st["duration"] = np.array([800.0 / c["rate"]])
        st["lum"] = torch.zeros((n, rows), dtype=torch.uint8, device="cuda")
        st["t"] = torch.zeros((n, rows), dtype=torch.float64, device="cuda")
        st["ratio"] = torch.zeros((n, rows), dtype=torch.float64, device="cuda")
        st["used"] = np.zeros(n, np.int32)
    elif kind == "lab":
        st["runs"], st["obs"] = _lab_runs(c)
    elif kind == "curves":
        st["theta"] = S.KINDS[c["curve"]].sample_params(c["sets"], np.random.default_rng(seed))
    elif kind == "glow":
        st["runs"], st["counts"] = run_array(_glow_runs(c)), _glow_counts(c, seed)
        points = int((427.0 + 8.0) / c["width"]) + 8
        st["curve"] = torch.zeros((c["runs"], points), dtype=torch.float64, device="cuda")
        st["lens"] = torch.zeros(c["runs"], dtype=torch.int32, device="cuda")
    elif kind == "infer":
        st["net"] = S.Network(_ctx(), max_batch=-(-c["batch"] // 64) * 64, params=_params(seed))
        st["x"] = _inputs(c["batch"], seed)
    elif kind == "train":
        st["net"] = S.Network(_ctx(), max_batch=c["batch"], params=_params(seed))
        st["x"] = _inputs(c["rows"], seed)
        st["t"] = _targets(st["x"])
        st["cfg"] = S.TrainConfig(epochs=1, batch=c["batch"], seed=seed)
    else:
        st["net"] = S.Network.load(_ctx(), WEIGHTS, max_batch=4096)
        y = S.denormalise(_targets(_inputs(1, seed)).cpu().numpy()[0])
        st["scale"] = 1e4 / y.max()
        st["y"] = np.random.default_rng(seed).poisson(y * st["scale"]).astype(np.float64)
    torch.cuda.current_stream().synchronize()
    return st


def run(st):
    c, kind = st["case"], st["kind"]
    if kind == "sweep":
        counts, live, _ = _ctx().run_fixed_dt(st["runs"], seed=st["seed"], n_bins=c["bins"])
        return {"counts": counts.view(np.int32), "live": live.view(np.int64)}
    if kind in ("decay", "large", "uneven"):
        st["plan"].launch(st["counts"].data_ptr(), st["live"].data_ptr())
        return {"counts": st["counts"], "live": st["live"]}
    if kind == "event":
        ctx = _ctx()
        ctx.check(ctx.lib.mcl_run_event(
            ctx.handle, st["runs"], 1, st["duration"].ctypes.data, C.c_uint64(st["seed"]), c["rows"],
            F_DEVICE_PTRS, st["lum"].data_ptr(), st["t"].data_ptr(), st["ratio"].data_ptr(),
            st["used"].ctypes.data, C.byref(Stats())), "mcl_run_event")
        return {"lum": st["lum"], "t": st["t"], "ratio": st["ratio"], "rows": st["used"]}
    if kind == "lab":
        ratio, status, _ = _ctx().run_lab(st["runs"], st["obs"], exact_fill=c["fill"], seed=st["seed"])
        return {"ratio": ratio, "status": status}
    if kind == "curves":
        return {"curves": S.KINDS[c["curve"]].mc_curves(_ctx(), st["theta"], n=c["electrons"],
                                                        sims=c["sims"], seed=st["seed"])}
    if kind == "glow":
        _ctx().glow_curve_device(st["runs"], st["counts"].data_ptr(), 4, st["counts"].shape[1], None,
                                 c["width"], 50.0, st["curve"].data_ptr(), st["curve"].shape[1],
                                 st["lens"].data_ptr())
        return {"curve": st["curve"], "lens": st["lens"]}
    if kind == "infer":
        return {"y": st["net"].forward(st["x"])}
    if kind == "train":
        r = S.train(st["net"], st["x"], st["t"], st["cfg"], log=None)
        return {"loss": r["loss"], "params": st["net"].get_params()}
    de = fit.NetworkDE(st["net"], st["y"], st["scale"], [0.1], fit.N_FIT, c["pop"], st["seed"])
    best = []
    for _ in range(c["gens"] // 25):          # the patience check of a fit: every 25 generations
        de.run(25)
        best.append(de.best()[1])
    x, f = de.population()
    de.close()
    return {"best": np.array(best, np.float32), "x": x, "f": f}


# ------------------------------------------------------------ work and exact values -------
def _live_steps(r):
    """Live electron-steps of one cluster's band decay (an upper figure where it tunnels)."""
    n0 = float(int(r.N_e * r.e_ratio_start))
    t = np.arange(int(r.n_steps)) * r.dt
    kT = r.k_b * (r.T_start + 273.15 + r.T_rate * t)
    x = np.minimum(r.s * np.exp(-np.minimum(r.E_cb / kT, 700.0)) * r.dt, 50.0)
    return n0 * float(np.exp(-np.concatenate([[0.0], np.cumsum(x)[:-1]])).sum())


def _mc_ops(runs):
    """28 integer and float operations per live electron-step (a quarter of a Philox4x32-10
    block, the rate's fma and the test) and 54 distances of 9 operations per electron's first
    nearest hole."""
    return sum(r.sims * (28.0 * _live_steps(r) + 486.0 * r.N_e * r.e_ratio_start) for r in runs)


def work(case):
    c = dict(case)
    kind = c["kind"]
    net = float(sum(a * b for a, b in zip(LAYERS[:-1], LAYERS[1:])))      # multiply-adds of a row
    if kind in ("sweep", "decay", "large"):
        rows = c["sims"] * (c.get("bins") or _runs(c)[0].n_steps)
        return {"bytes": 4.0 * rows + 8.0 * c["sims"], "flops": _mc_ops(_runs(c))}
    if kind == "uneven":
        some = W.uneven_sweep(min(c["sets"], 500), seed=1, n_steps=c["steps"])
        return {"bytes": (4.0 * c["bins"] + 8.0) * c["sets"],
                "flops": _mc_ops(some) * c["sets"] / len(some)}
    if kind == "event":
        # two float64 operations per live electron of a recombination step, half of them live
        return {"bytes": 17.0 * c["sims"] * c["rows"], "flops": c["sims"] * float(c["electrons"]) ** 2}
    if kind == "lab":
        n = c["sets"] * c["rows"] * c["sims"]
        return {"bytes": 12.0 * n, "flops": 2.0 * 250 * 60 * n}            # ~250 events of ~60 electrons
    if kind == "curves":
        k = S.KINDS[c["curve"]]
        runs = [k.run(t, c["electrons"], c["sims"]) for t in k.sample_params(24, np.random.default_rng(1))]
        return {"bytes": 8.0 * S.N_BINS * c["sets"], "flops": _mc_ops(runs) * c["sets"] / len(runs)}
    if kind == "glow":
        n = float(c["runs"] * c["sims"] * c["steps"])
        return {"bytes": 4.0 * n + 8.0 * c["runs"] * 400.0 / c["width"], "flops": n}
    if kind == "infer":
        return {"bytes": 4.0 * c["batch"] * (S.N_IN + S.N_BINS) + 2.0 * net, "flops": 2.0 * net * c["batch"]}
    if kind == "train":
        steps = c["rows"] // c["batch"]
        return {"bytes": steps * (4.0 * c["batch"] * (S.N_IN + S.N_BINS) + 28.0 * net),
                "flops": steps * 6.0 * net * c["batch"]}
    return {"bytes": 4.0 * c["pop"] * 6 + 2.0 * net, "flops": 2.0 * net * c["pop"] * (c["gens"] + 1)}


def _layers(flat):
    out, o = [], 0
    p = torch.from_numpy(flat).cuda().double()
    for k, n in zip(LAYERS[:-1], LAYERS[1:]):
        out.append([p[o:o + n * k].view(n, k).clone(), p[o + n * k:o + n * k + n].clone()])
        o += n * k + n
    return out


def _net64(layers, x):
    """Activations of every layer in float64: [(input, pre-activation)]."""
    acts = []
    for i, (w, b) in enumerate(layers):
        z = x @ w.t() + b
        acts.append((x, z))
        x = z if i == len(layers) - 1 else z * torch.sigmoid(z)
    return acts


def _exact_train(c, seed):
    cfg = S.TrainConfig(epochs=1, batch=c["batch"], seed=seed)
    x = _inputs(c["rows"], seed)
    t = _targets(x).double()
    x = x.double()
    layers = _layers(_params(seed))
    flat = [p for layer in layers for p in layer]
    m = [torch.zeros_like(p) for p in flat]
    v = [torch.zeros_like(p) for p in flat]
    n_steps = c["rows"] // c["batch"]
    perm = torch.randperm(c["rows"], generator=torch.Generator(device="cpu").manual_seed(seed)).cuda()
    losses = []
    for k in range(n_steps):
        idx = perm[k * c["batch"]:(k + 1) * c["batch"]]
        acts = _net64(layers, x[idx])
        d = acts[-1][1] - t[idx]
        losses.append((d * d).mean())
        g = d * (2.0 / d.numel())
        grads = []
        for i in range(len(layers) - 1, -1, -1):
            grads = [g.t() @ acts[i][0], g.sum(0)] + grads
            if i > 0:
                z = acts[i - 1][1]
                s = torch.sigmoid(z)
                g = (g @ layers[i][0]) * (s * (1.0 + z * (1.0 - s)))
        step = k + 1
        if step <= cfg.warmup_steps:
            lr = cfg.lr * step / cfg.warmup_steps
        else:
            f = (step - cfg.warmup_steps) / max(1, n_steps - cfg.warmup_steps)
            lr = cfg.lr_min + 0.5 * (cfg.lr - cfg.lr_min) * (1.0 + math.cos(math.pi * f))
        for p, gr, a, b in zip(flat, grads, m, v):
            p.mul_(1.0 - lr * cfg.weight_decay)
            a.mul_(cfg.beta1).add_(gr, alpha=1.0 - cfg.beta1)
            b.mul_(cfg.beta2).addcmul_(gr, gr, value=1.0 - cfg.beta2)
            p.sub_(lr / (1.0 - cfg.beta1 ** step) * a /
                   (b.sqrt() / math.sqrt(1.0 - cfg.beta2 ** step) + cfg.eps))
    return {"loss": torch.stack(losses), "params": torch.cat([p.reshape(-1) for p in flat])}


def _exact_glow(c, seed):
    counts = _glow_counts(c, seed).cpu().numpy().reshape(c["runs"], c["sims"], c["steps"])
    points = int((427.0 + 8.0) / c["width"]) + 8
    out = np.zeros((c["runs"], points))
    r0 = _glow_runs(dict(c, runs=1))[0]
    T = r0.T_start + r0.T_rate * (np.arange(1, c["steps"] + 1, dtype=np.float64) * r0.dt)
    bins = np.arange(0, T.max() + c["width"], c["width"])
    k = max(1, int(50.0 / c["width"]))
    for r in range(c["runs"]):
        h, _ = np.histogram(T, bins=bins, weights=counts[r].mean(axis=0))
        y = np.convolve(h / c["width"], np.ones(k) / k, "valid")
        out[r, :y.size] = y
    return {"curve": out, "lens": None}


def exact(case, seed):
    c = dict(case)
    if c["kind"] == "infer":
        return {"y": _net64(_layers(_params(seed)), _inputs(c["batch"], seed).double())[-1][1]}
    if c["kind"] == "train":
        return _exact_train(c, seed)
    if c["kind"] == "glow":
        return _exact_glow(c, seed)
    return None
