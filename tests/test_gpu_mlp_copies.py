"""The BF16 copies of the weights that a training step leaves behind (row-major, and the fragments
of W and W^T): forward and gradient of a trained network equal, bit for bit, those of a new
network given its parameters, whose copies another kernel writes."""
import pytest

from mcluminescence_amd import surrogate as S
from mcluminescence_amd._abi import AdamW

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_out", [256, 512])
def test_copies_follow_the_steps(gpu_ctx, n_out):
    import torch
    print(f"weight copies: {n_out} outputs", flush=True)
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.rand((512, 6), generator=g, device="cuda") * 2 - 1
    t = torch.rand((512, n_out), generator=g, device="cuda")
    idx = torch.randperm(512, generator=g, device="cuda")[:320].to(torch.int32)
    net = S.Network(gpu_ctx, n_out=n_out, max_batch=512, seed=8)
    # large steps, so that every weight's BF16 copy changes
    for step in range(1, 4):
        net.train_step(x, t, idx, AdamW(0.05, 0.9, 0.999, 1e-8, 0.0, step))
    new = S.Network(gpu_ctx, n_out=n_out, max_batch=512, params=net.get_params())
    try:
        la, ga = net.grad(x, t, idx)
        lb, gb = new.grad(x, t, idx)
        assert la == lb
        assert torch.equal(ga, gb)
        ya, yb = net.forward(x), new.forward(x)
        assert torch.equal(ya, yb)
        gpu_ctx.tune_set("mlp_fused", 0)          # and the row-major copies
        try:
            assert torch.equal(net.forward(x), ya)
        finally:
            gpu_ctx.tune_set("mlp_fused", 1)
    finally:
        net.close()
        new.close()
