"""Training in two kernels against training layer by layer (a network made with the mlp_fused knob
at 0, and the form of every other shape): gradients, weights after several AdamW steps and outputs
bit for bit, at batches summed in one, two, four and eight parts; and the layered form of
other shapes against the oracle."""
import numpy as np
import pytest

from mcluminescence_amd import surrogate as S
from mcluminescence_amd._abi import AdamW
from oracle import mlp_oracle as O

pytestmark = pytest.mark.gpu


def _layered(ctx, **kw):
    ctx.tune_set("mlp_fused", 0)
    try:
        return S.Network(ctx, **kw)
    finally:
        ctx.tune_set("mlp_fused", 1)


def _data(n_out, rows, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.rand((rows, 6), generator=g, device="cuda") * 2 - 1
    t = torch.rand((rows, n_out), generator=g, device="cuda")
    return g, x, t


@pytest.mark.parametrize("n_out", [256, 512])
@pytest.mark.parametrize("batch", [64, 128, 192, 256, 384, 512, 640, 1024, 4160])
def test_two_kernels_equal_the_layers(gpu_ctx, n_out, batch):
    import torch
    print(f"training forms: {n_out} outputs, batch {batch}", flush=True)
    g, x, t = _data(n_out, 2 * batch, batch)
    idx = torch.randperm(2 * batch, generator=g, device="cuda")[:batch].to(torch.int32)
    two = S.Network(gpu_ctx, n_out=n_out, max_batch=batch, seed=5)
    lay = _layered(gpu_ctx, n_out=n_out, max_batch=batch, seed=5)
    try:
        for rows in (idx, None):
            xr, tr = (x, t) if rows is not None else (x[:batch], t[:batch])
            la, ga = two.grad(xr, tr, rows)
            lb, gb = lay.grad(xr, tr, rows)
            assert torch.equal(ga, gb)
            # (the losses add the same squares in different orders: at most a rounding of each
            # of the additions a partial sum takes)
            assert abs(la - lb) <= 1e-5 * lb
        for step in range(1, 6):
            hp = AdamW(2e-3, 0.9, 0.999, 1e-8, 0.01, step)
            two.train_step(x, t, idx, hp)
            lay.train_step(x, t, idx, hp)
        np.testing.assert_array_equal(two.get_params(), lay.get_params())
        ga, gb = two.grad(x, t, idx)[1], lay.grad(x, t, idx)[1]
        assert torch.equal(ga, gb)
        assert torch.equal(two.forward(x[:batch]), lay.forward(x[:batch]))
    finally:
        two.close()
        lay.close()


@pytest.mark.parametrize("d", [O.Desc(6, 128, 1, 128), O.Desc(6, 128, 2, 256), O.Desc(5, 512, 3, 256),
                               O.Desc(6, 512, 5, 512), O.Desc(6, 256, 4, 256)])
def test_layered_shapes(gpu_ctx, d):
    import torch
    print(f"layered training: {d}", flush=True)
    p0 = O.init_params(d, seed=6)
    net = S.Network(gpu_ctx, d.n_in, d.n_hidden, d.n_hidden_layers, d.n_out, 256, params=p0)
    rng = np.random.default_rng(7)
    x = rng.uniform(-1, 1, (256, d.n_in)).astype(np.float32)
    t = rng.uniform(0, 1, (256, d.n_out)).astype(np.float32)
    xt, tt = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    idx = torch.arange(256, dtype=torch.int32, device="cuda")
    try:
        loss, g = net.grad(xt, tt)
        g = g.cpu().numpy()
        lq, gq = O.loss_grad(p0, d, x, t, quantize=True)
        assert abs(loss - lq) / lq < 1e-3
        G, Q = O.split_flat(g, d), O.split_flat(gq, d)
        for k in G:
            rel = float(np.linalg.norm(G[k] - Q[k]) / np.linalg.norm(Q[k]))
            assert rel < 2e-2, f"{k}: {rel:.2e}"
        m = v = np.zeros_like(g, dtype=np.float64)
        p = p0
        for step in range(1, 4):
            _, g = net.grad(xt, tt)
            g = g.cpu().numpy().astype(np.float64)
            net.train_step(xt, tt, idx, AdamW(1e-3, 0.9, 0.999, 1e-8, 0.01, step))
            ref, m, v = O.adamw(p, g, m, v, lr=1e-3, weight_decay=0.01, step=step)
            p = net.get_params()
            np.testing.assert_allclose(p, ref, rtol=1e-5, atol=1e-7)
        # the next forward uses the weights of the last step
        y = net.forward(xt).cpu().numpy()
        yq, _ = O.forward(p, d, x, quantize=True)
        assert np.linalg.norm(y - yq) / np.linalg.norm(yq) < 5e-3
    finally:
        net.close()
