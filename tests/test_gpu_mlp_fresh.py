"""A network straight from mcl_mlp_create, before any mcl_mlp_set_params: its parameters are zeros,
and the forward, the gradient and an AdamW step are those of zeros, in both forms of the kernels,
whatever the device memory held before."""
import ctypes as C

import numpy as np
import pytest

from mcluminescence_amd import surrogate as S
from mcluminescence_amd._abi import AdamW, MlpDesc

pytestmark = pytest.mark.gpu


def _dirty_memory(ctx, n_out):
    """Freed allocations of a network's sizes that hold weights, and freed blocks of NaN."""
    import torch
    blocks = [torch.full((1 << 20,), float("nan"), device="cuda") for _ in range(64)]
    torch.cuda.synchronize()
    del blocks
    torch.cuda.empty_cache()
    for _ in range(2):
        S.Network(ctx, n_out=n_out, max_batch=256, seed=3).close()


@pytest.mark.parametrize("n_out", [256, 512])
@pytest.mark.parametrize("fused", [1, 0])
def test_zeros_until_parameters_are_set(gpu_ctx, n_out, fused):
    import torch
    print(f"fresh network: {n_out} outputs, mlp_fused {fused}", flush=True)
    _dirty_memory(gpu_ctx, n_out)
    lib = gpu_ctx.lib
    desc = MlpDesc(6, 512, 4, n_out, 256)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand((256, 6), generator=g, device="cuda") * 2 - 1
    t = torch.rand((256, n_out), generator=g, device="cuda")
    idx = torch.arange(256, dtype=torch.int32, device="cuda")
    y = torch.full((256, n_out), 7.0, device="cuda")
    h = C.c_void_p()
    gpu_ctx.tune_set("mlp_fused", fused)
    try:
        gpu_ctx.check(lib.mcl_mlp_create(gpu_ctx.handle, C.byref(desc), C.byref(h)), "mcl_mlp_create")
        n = int(lib.mcl_mlp_param_count(h))
        grad = torch.full((n,), 7.0, device="cuda")
        loss = torch.zeros(1, device="cuda")
        torch.cuda.synchronize()

        def call(name, *args):
            gpu_ctx.check(getattr(lib, name)(h, *args), name)
            torch.cuda.synchronize()

        params = np.full(n, 7.0, np.float32)
        call("mcl_mlp_get_params", params.ctypes.data)
        assert not params.any()
        call("mcl_mlp_forward", x.data_ptr(), 256, y.data_ptr())
        assert torch.equal(y, torch.zeros_like(y))
        # y = 0 and silu(0) = 0: only the output biases have a gradient
        call("mcl_mlp_grad", x.data_ptr(), t.data_ptr(), None, 256, grad.data_ptr(), loss.data_ptr())
        want = -(2.0 / t.numel()) * t.double().sum(0)
        assert not grad[:-n_out].any()
        torch.testing.assert_close(grad[-n_out:].double(), want, rtol=2 ** -8, atol=0)
        assert abs(float(loss) - float((t.double() ** 2).mean())) < 1e-5
        hp = AdamW(1e-3, 0.9, 0.999, 1e-8, 0.0, 1)
        call("mcl_mlp_train_step", x.data_ptr(), t.data_ptr(), idx.data_ptr(), 256, C.byref(hp),
             loss.data_ptr())
        call("mcl_mlp_get_params", params.ctypes.data)
        assert not params[:-n_out].any()
        np.testing.assert_allclose(params[-n_out:], 1e-3, rtol=1e-4)
        # and the copies the next forward reads follow the step
        call("mcl_mlp_forward", x.data_ptr(), 256, y.data_ptr())
        np.testing.assert_array_equal(y.cpu().numpy(), np.tile(params[-n_out:], (256, 1)))
    finally:
        gpu_ctx.tune_set("mlp_fused", 1)
        if h.value:
            lib.mcl_mlp_destroy(h)
