"""A plan's work figures (mcl_plan_work) are the same for every launch, with one and with several
waves a cluster, in LDS and in scratch memory."""
import pytest

from mcluminescence_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", [1, 2, 4, 8])
@pytest.mark.parametrize("global_memory", [0, 1])
def test_same_work_every_launch(gpu_ctx, waves, global_memory):
    import torch
    print(f"work: {waves} waves, global_memory {global_memory}", flush=True)
    runs = [W.single_trap(1.3, 1e12, 4e9, 1e23, n, T_start_K=300.0, T_rate=1.0, dt=0.1, n_steps=4000,
                          sims=24) for n in (150, 600)]
    gpu_ctx.tune_set("waves_per_cluster", waves)
    gpu_ctx.tune_set("global_memory", global_memory)
    try:
        plan = gpu_ctx.plan(runs)
    finally:
        gpu_ctx.tune_set("waves_per_cluster", 0)
        gpu_ctx.tune_set("global_memory", 0)
    counts = torch.zeros((48, 4000), dtype=torch.int32, device="cuda")
    rows = set()
    for _ in range(6):
        plan.launch(counts.data_ptr())
        w = plan.work()
        rows.add((w.live_electron_steps, w.distance_evals, w.recombinations, w.cluster_steps))
    plan.close()
    assert len(rows) == 1
