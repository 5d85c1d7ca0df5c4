"""The fused inference and training kernels at the batch sizes where they can go wrong: one
workgroup, batches around the change from 32 to 64 rows a workgroup, and batches whose
weight gradients are summed in one, two, four and eight parts; 256 and 512 outputs."""
import numpy as np
import pytest

from mcluminescence_amd import surrogate as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[256, 512])
def net(request, gpu_ctx):
    n = S.Network(gpu_ctx, n_out=request.param, max_batch=8320, seed=4)
    yield n
    n.close()


@pytest.mark.parametrize("batch", [64, 320, 8128, 8192, 8256, 8320])
def test_fused_inference_equals_layered(net, gpu_ctx, batch):
    import torch
    print(f"inference: {net.desc.n_out} outputs, batch {batch}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(batch)
    x = torch.rand((batch, 6), generator=g, device="cuda") * 2 - 1
    y = net.forward(x)
    gpu_ctx.tune_set("mlp_fused", 0)
    try:
        ref = net.forward(x)
    finally:
        gpu_ctx.tune_set("mlp_fused", 1)
    torch.testing.assert_close(y, ref, rtol=0, atol=0)


@pytest.mark.parametrize("batch", [64, 128, 192, 256, 512, 640, 1024, 4160])
def test_gradient_matches_float64(net, batch):
    # BF16 weights, activations and errors against the exact network: the relative error of
    # a layer's gradient is that of 2^-9 roundings through five layers (0.4 % measured for
    # the layered kernels at batch 4096); small batches average fewer rows
    import torch
    print(f"gradient: {net.desc.n_out} outputs, batch {batch}", flush=True)
    n_out = net.desc.n_out
    g = torch.Generator(device="cuda").manual_seed(batch)
    x = torch.rand((2 * batch, 6), generator=g, device="cuda") * 2 - 1
    t = torch.rand((2 * batch, n_out), generator=g, device="cuda")
    idx = torch.randperm(2 * batch, generator=g, device="cuda")[:batch].to(torch.int32)
    loss, grad = net.grad(x, t, idx)
    p = torch.from_numpy(net.get_params()).cuda().double()
    dims = [6, 512, 512, 512, 512, n_out]
    layers, o = [], 0
    for k, n in zip(dims[:-1], dims[1:]):
        layers.append((p[o:o + n * k].view(n, k), p[o + n * k:o + n * k + n]))
        o += n * k + n
    a, zs, acts = x[idx.long()].double(), [], []
    for i, (w, b) in enumerate(layers):
        acts.append(a)
        z = a @ w.t() + b
        zs.append(z)
        a = z if i == 4 else z * torch.sigmoid(z)
    d = a - t[idx.long()].double()
    assert abs(loss - float((d * d).mean())) <= 1e-2 * float((d * d).mean())
    e = d * (2.0 / d.numel())
    want = []
    for i in range(4, -1, -1):
        want = [(e.t() @ acts[i]).reshape(-1), e.sum(0)] + want
        if i:
            s = torch.sigmoid(zs[i - 1])
            e = (e @ layers[i][0]) * (s * (1 + zs[i - 1] * (1 - s)))
    o = 0
    for i, v in enumerate(want):
        got = grad[o:o + v.numel()].double()
        o += v.numel()
        rel = float((got - v).norm() / v.norm())
        assert rel < 2e-2, f"part {i}: {rel:.2e}"
    assert o == grad.numel()
