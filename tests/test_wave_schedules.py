"""The fixed-dt kernels with several waves a cluster, whatever order the waves run in: their own
source on the CPU (wave_model), with one wave far behind or far ahead of the others, or in a
random order.  The workgroup barriers must meet at the same place in every wave, and counts and
live steps must be those of the replay harness; the work counted must not depend on the order."""
import numpy as np
import pytest

import wave_model as wm
from mcluminescence_amd import workloads as W
from oracle import orc


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    return wm.Model(tmp_path_factory.mktemp("wave_model") / "wave_model.so")


def _runs(kind):
    if kind == "sparse":          # most windows have no event, then some have a few
        return [W.single_trap(1.3, 1e12, 4e9, 1e23, n, T_start_K=300.0, T_rate=1.0, dt=0.1,
                              n_steps=4000, sims=s) for n, s in ((5, 2), (130, 1))]
    if kind == "tail":            # an isothermal decay down to its last electrons
        return [W.single_trap(1.4, 1e13, 4e9, 1e23, 70, T_start_K=480.0, T_rate=0.0, dt=0.5,
                              n_steps=3000, sims=2)]
    if kind == "many":            # steps with more than 64 candidates, fewer holes than electrons
        hot = W.single_trap(1.4, 1e13, 4e9, 1e23, 400, T_start_K=548.0, T_rate=0.0, dt=0.5,
                            n_steps=70, sims=1)
        few = W.single_trap(1.4, 1e13, 4e9, 1e23, 150, T_start_K=700.0, T_rate=0.0, dt=0.5,
                            n_steps=70, sims=1)
        few.holes = 50.0
        return [hot, few]
    r = W.tunnelling_tl12(sims=1, n=300, T_rate=5.0)[0]
    r.rho_prime, r.n_steps, r.dt = 3e-3, 200, 0.8
    r.E_loc_1, r.E_loc_2, r.Retrap = 1.1, 1.3, 0.4
    return [r]


def _schedules(waves):
    yield wm.IN_TURN, 0
    for w in {0, 1, waves - 1}:
        yield wm.behind(w), 0
        yield wm.ahead(w), 0
    for seed in range(3):
        yield wm.SHUFFLED, seed


@pytest.mark.parametrize("kind", ["sparse", "tail", "many", "two_channel"])
@pytest.mark.parametrize("waves", [1, 2, 4, 8])
@pytest.mark.parametrize("form", [wm.LDS, wm.SCRATCH, wm.SCRATCH_ALL])
def test_any_order_of_the_waves(model, kind, waves, form):
    runs = _runs(kind)
    ref, ref_live = orc.run_fixed_dt(runs, threads=8)
    for schedule, seed in _schedules(waves):
        for persistent in ([False, True] if form == wm.LDS and schedule < 100 else [True]):
            what = f"schedule {schedule} (seed {seed}), persistent {persistent}"
            got, live, _, error = model.run(runs, waves, form=form, persistent=persistent,
                                            schedule=schedule, schedule_seed=seed)
            assert error == "", f"{what}: {error}"
            np.testing.assert_array_equal(got, ref, err_msg=what)
            np.testing.assert_array_equal(live, ref_live, err_msg=what)


@pytest.mark.parametrize("waves", [1, 4])
def test_wider_blocks(model, waves):
    runs = [W.single_trap(1.3, 1e12, 4e9, 1e23, 250, T_start_K=440.0, T_rate=1.0, dt=0.5,
                          n_steps=200, sims=1)]
    ref, ref_live = orc.run_fixed_dt(runs, n_bins=13, threads=8)
    for hpc in (2.0, 0.05):       # grids of 6 and of 20 cells an axis
        for schedule, seed in _schedules(waves):
            got, live, _, error = model.run(runs, waves, n_bins=13, wide=True, holes_per_cell=hpc,
                                            schedule=schedule, schedule_seed=seed)
            assert error == ""
            np.testing.assert_array_equal(got, ref)
            np.testing.assert_array_equal(live, ref_live)


@pytest.mark.parametrize("kind", ["sparse", "tail", "many", "two_channel"])
@pytest.mark.parametrize("waves", [2, 4, 8])
@pytest.mark.parametrize("form", [wm.LDS, wm.SCRATCH_ALL])
def test_work_does_not_depend_on_the_order(model, kind, waves, form):
    runs = _runs(kind)
    ref = None
    for schedule, seed in _schedules(waves):
        _, _, work, error = model.run(runs, waves, form=form, persistent=form != wm.LDS,
                                      schedule=schedule, schedule_seed=seed)
        assert error == ""
        if ref is None:
            ref = work
        np.testing.assert_array_equal(work, ref, err_msg=f"schedule {schedule} (seed {seed})")
