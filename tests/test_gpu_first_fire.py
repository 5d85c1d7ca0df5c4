"""The fixed-dt kernels' first-fire windows at the sizes where they can go wrong, bit-exact
against the CPU replay harness, which steps through every step.

Edges: runs that end inside, on and just past a 64-step window and an 8-step sub-window;
rows at, below and above the live count that switches the scan from 16 lanes an electron
to one; clusters of one electron, one row and one slot more; steps with 64 and 65
candidates (one wave, then all of them); grids below and at the size from which
inconclusive searches take wider blocks; each for ramps, isothermal and two-channel
runs and one to eight waves a cluster."""
import numpy as np
import pytest

from mcluminescence_amd import workloads as W
from oracle import orc

pytestmark = pytest.mark.gpu


def _physics(kind, n, n_steps, sims):
    if kind == "ramp":            # the whole glow peak within the run
        return W.single_trap(1.3, 1e12, 4e9, 1e23, n, T_start_K=430.0, T_rate=1.0,
                             dt=120.0 / n_steps, n_steps=n_steps, sims=sims)
    if kind == "cooling":         # the thresholds fall through the window
        return W.single_trap(1.3, 1e12, 4e9, 1e23, n, T_start_K=500.0, T_rate=-1.0,
                             dt=60.0 / n_steps, n_steps=n_steps, sims=sims)
    if kind == "iso":
        return W.single_trap(1.4, 1e13, 4e9, 1e23, n, T_start_K=500.0, T_rate=0.0,
                             dt=40.0 / n_steps, n_steps=n_steps, sims=sims)
    r = W.tunnelling_tl12(sims=sims, n=n, T_rate=5.0)[0]
    r.rho_prime, r.n_steps, r.dt = 3e-3, n_steps, 160.0 / n_steps
    r.E_loc_1, r.E_loc_2, r.Retrap = 1.1, 1.3, 0.4
    return r


def _same(ctx, runs, waves, n_bins=None):
    ctx.tune_set("waves_per_cluster", waves)
    try:
        got, live, _ = ctx.run_fixed_dt(runs, n_bins=n_bins)
    finally:
        ctx.tune_set("waves_per_cluster", 0)
    ref, ref_live = orc.run_fixed_dt(runs, n_bins=n_bins, threads=8)
    np.testing.assert_array_equal(got, ref)
    np.testing.assert_array_equal(live, ref_live)


@pytest.mark.parametrize("kind", ["ramp", "cooling", "iso", "two_channel"])
@pytest.mark.parametrize("waves", [1, 2, 8])
def test_window_edges(gpu_ctx, kind, waves):
    print(f"window edges: {kind}, {waves} waves", flush=True)
    for n_steps in (1, 3, 7, 8, 9, 63, 64, 65, 72, 127, 129, 257):
        runs = [_physics(kind, n, n_steps, 2) for n in (1, 16, 17, 64, 65, 200)]
        _same(gpu_ctx, runs, waves)
    _same(gpu_ctx, [_physics(kind, 150, 130, 3)], waves, n_bins=13)
    _same(gpu_ctx, [_physics(kind, 150, 130, 3)], waves, n_bins=47)


@pytest.mark.parametrize("waves", [1, 4])
@pytest.mark.parametrize("n", [64, 65, 130, 700])
def test_steps_with_many_candidates(gpu_ctx, n, waves):
    # p = 1 at 700 K: every electron is a candidate of the first step
    print(f"many candidates: {n} electrons, {waves} waves", flush=True)
    hot = W.single_trap(1.4, 1e13, 4e9, 1e23, n, T_start_K=700.0, T_rate=0.0, dt=0.5, n_steps=70,
                        sims=3)
    few = W.single_trap(1.4, 1e13, 4e9, 1e23, n, T_start_K=700.0, T_rate=0.0, dt=0.5, n_steps=70,
                        sims=3)
    few.holes = max(1.0, n / 3.0)          # fewer holes than electrons
    warm = W.single_trap(1.4, 1e13, 4e9, 1e23, n, T_start_K=548.0, T_rate=0.0, dt=0.5, n_steps=70,
                         sims=3)           # p = 0.5
    _same(gpu_ctx, [hot, few, warm], waves)


@pytest.mark.parametrize("n", [842, 844, 1300])
@pytest.mark.parametrize("hpc", [2.0, 1.0])
def test_grids_around_the_wide_search(gpu_ctx, n, hpc):
    # 842 and 844 core holes make 1454 and 1458 holes: grids of 8 and 9 cells an axis
    print(f"wide grids: {n} electrons, {hpc} holes per cell", flush=True)
    gpu_ctx.tune_set("holes_per_cell", hpc)
    try:
        _same(gpu_ctx, [_physics("ramp", n, 300, 2), _physics("two_channel", n, 100, 2)], 4)
    finally:
        gpu_ctx.tune_set("holes_per_cell", 2)
