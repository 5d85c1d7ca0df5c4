"""The first-fire windows' edges in the kernels' other forms, bit-exact against the CPU replay: the
global-memory form, the build for large grids (blocks of 5 and of 9 cells), each with one to
eight waves a cluster, one workgroup a cluster and persistent."""
import numpy as np
import pytest

from mcluminescence_amd import workloads as W
from mcluminescence_amd._abi import F_PERSISTENT
from oracle import orc

pytestmark = pytest.mark.gpu


def _physics(kind, n, n_steps, sims):
    if kind == "ramp":
        return W.single_trap(1.3, 1e12, 4e9, 1e23, n, T_start_K=430.0, T_rate=1.0,
                             dt=120.0 / n_steps, n_steps=n_steps, sims=sims)
    if kind == "cooling":
        return W.single_trap(1.3, 1e12, 4e9, 1e23, n, T_start_K=500.0, T_rate=-1.0,
                             dt=60.0 / n_steps, n_steps=n_steps, sims=sims)
    if kind == "iso":
        return W.single_trap(1.4, 1e13, 4e9, 1e23, n, T_start_K=500.0, T_rate=0.0,
                             dt=40.0 / n_steps, n_steps=n_steps, sims=sims)
    if kind == "sparse":          # windows without an event between those with a few
        return W.single_trap(1.3, 1e12, 4e9, 1e23, n, T_start_K=300.0, T_rate=1.0, dt=0.1,
                             n_steps=n_steps, sims=sims)
    r = W.tunnelling_tl12(sims=sims, n=n, T_rate=5.0)[0]
    r.rho_prime, r.n_steps, r.dt = 3e-3, n_steps, 160.0 / n_steps
    r.E_loc_1, r.E_loc_2, r.Retrap = 1.1, 1.3, 0.4
    return r


def _same(ctx, runs, waves, knobs, flags=0, n_bins=None):
    for k, v in dict(knobs, waves_per_cluster=waves).items():
        ctx.tune_set(k, v)
    try:
        got, live, _ = ctx.run_fixed_dt(runs, n_bins=n_bins, flags=flags)
    finally:
        ctx.tune_set("waves_per_cluster", 0)
        ctx.tune_set("global_memory", 0)
        ctx.tune_set("holes_per_cell", 2)
    ref, ref_live = orc.run_fixed_dt(runs, n_bins=n_bins, threads=8)
    np.testing.assert_array_equal(got, ref)
    np.testing.assert_array_equal(live, ref_live)


@pytest.mark.parametrize("kind", ["ramp", "cooling", "iso", "two_channel"])
@pytest.mark.parametrize("waves", [1, 2, 8])
def test_window_edges_in_global_memory(gpu_ctx, kind, waves):
    print(f"window edges in global memory: {kind}, {waves} waves", flush=True)
    for n_steps in (1, 3, 7, 8, 9, 63, 64, 65, 72, 127, 129, 257):
        runs = [_physics(kind, n, n_steps, 2) for n in (1, 16, 17, 64, 65, 200)]
        _same(gpu_ctx, runs, waves, {"global_memory": 1})
    _same(gpu_ctx, [_physics(kind, 150, 130, 3)], waves, {"global_memory": 1}, n_bins=47)


@pytest.mark.parametrize("waves", [1, 4])
@pytest.mark.parametrize("n", [64, 65, 130, 700])
def test_many_candidates_in_global_memory(gpu_ctx, n, waves):
    print(f"many candidates in global memory: {n} electrons, {waves} waves", flush=True)
    hot = W.single_trap(1.4, 1e13, 4e9, 1e23, n, T_start_K=700.0, T_rate=0.0, dt=0.5, n_steps=70,
                        sims=3)
    few = W.single_trap(1.4, 1e13, 4e9, 1e23, n, T_start_K=700.0, T_rate=0.0, dt=0.5, n_steps=70,
                        sims=3)
    few.holes = max(1.0, n / 3.0)
    warm = W.single_trap(1.4, 1e13, 4e9, 1e23, n, T_start_K=548.0, T_rate=0.0, dt=0.5, n_steps=70,
                         sims=3)
    _same(gpu_ctx, [hot, few, warm], waves, {"global_memory": 1})


@pytest.mark.parametrize("waves", [1, 2, 4, 8])
@pytest.mark.parametrize("flags", [0, F_PERSISTENT])
@pytest.mark.parametrize("global_memory", [0, 1])
def test_grids_on_both_sides_of_the_wide_build(gpu_ctx, waves, flags, global_memory):
    # 300 electrons: 518 holes in 6 cells an axis; 842 and 844 core holes make 1454 and 1458 holes, 8
    # and 9 cells an axis; at 0.25 holes a cell 1382 holes (800 electrons) take 17 or more
    print(f"grids: {waves} waves, flags {flags}, global_memory {global_memory}", flush=True)
    for n, hpc in ((300, 2.0), (842, 2.0), (844, 2.0), (800, 0.25)):
        runs = [_physics("ramp", n, 200, 2), _physics("two_channel", n, 100, 1)]
        _same(gpu_ctx, runs, waves, {"global_memory": global_memory, "holes_per_cell": hpc}, flags)


@pytest.mark.parametrize("waves", [1, 2, 4, 8])
@pytest.mark.parametrize("flags", [0, F_PERSISTENT])
def test_windows_without_events(gpu_ctx, waves, flags):
    print(f"sparse windows: {waves} waves, flags {flags}", flush=True)
    runs = [_physics("sparse", n, 4000, 4) for n in (1, 5, 70, 130)]
    for global_memory in (0, 1):
        _same(gpu_ctx, runs, waves, {"global_memory": global_memory}, flags)
