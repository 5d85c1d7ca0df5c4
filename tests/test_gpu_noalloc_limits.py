"""The allocation-free entry point takes the cluster sizes that mcl_cluster_limits counts (16
bytes an electron), whatever its layout takes."""
import pytest

from mcluminescence_amd import workloads as W
from mcluminescence_amd._abi import MclError

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,accepted", [(3400, True), (3700, False)])
def test_cluster_sizes(gpu_ctx, n, accepted):
    import torch
    runs = [W.single_trap(1.3, 1e12, 4e9, 1e23, n, T_start_K=300.0, T_rate=1.0, dt=0.1, n_steps=64,
                          sims=1)]
    counts = torch.zeros((1, 64), dtype=torch.int32, device="cuda")
    if accepted:
        gpu_ctx.run_fixed_dt_noalloc(runs, counts.data_ptr())
    else:
        with pytest.raises(MclError):
            gpu_ctx.run_fixed_dt_noalloc(runs, counts.data_ptr())
