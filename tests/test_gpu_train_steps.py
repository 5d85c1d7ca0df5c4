"""train() takes its steps through Network.train_step, a subclass's own included, within one
handshake of the streams an epoch, and the context is back on its own stream after each."""
import numpy as np
import pytest

from mcluminescence_amd import surrogate as S

pytestmark = pytest.mark.gpu


class Counting(S.Network):
    steps = 0
    fail_at = 0
    other = None

    def train_step(self, x, t, idx, hp, loss_out=None):
        self.steps += 1
        if self.other is not None:       # another network of the same context, between the steps
            self.other.forward(x[:256])
        if self.steps == self.fail_at:
            raise RuntimeError("stopped by the subclass")
        super().train_step(x, t, idx, hp, loss_out)


def test_train_calls_train_step(gpu_ctx):
    import torch
    print("train() through a subclass's train_step", flush=True)
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.rand((1024, 6), generator=g, device="cuda") * 2 - 1
    t = torch.rand((1024, 256), generator=g, device="cuda")
    cfg = S.TrainConfig(epochs=2, batch=256, warmup_steps=2)
    plain = S.Network(gpu_ctx, max_batch=256, seed=1)
    own = Counting(gpu_ctx, max_batch=256, seed=1)
    try:
        own.other = S.Network(gpu_ctx, max_batch=256, seed=2)
        a = S.train(plain, x, t, cfg, log=None)
        b = S.train(own, x, t, cfg, log=None)
        assert own.steps == 8
        np.testing.assert_array_equal(a["loss"], b["loss"])
        np.testing.assert_array_equal(plain.get_params(), own.get_params())
        calls = []
        patched = S.Network(gpu_ctx, max_batch=256, seed=1)
        step = patched.train_step
        patched.train_step = lambda *args: (calls.append(args[4]), step(*args))
        S.train(patched, x, t, cfg, log=None)
        assert len(calls) == 8
        np.testing.assert_array_equal(plain.get_params(), patched.get_params())
        patched.close()
        own.fail_at = 10
        with pytest.raises(RuntimeError, match="stopped"):
            S.train(own, x, t, cfg, log=None)
        # later calls make their own handshake again
        assert not own._entered
        y = own.forward(x[:256])
        plain.set_params(own.get_params())
        assert torch.equal(plain.forward(x[:256]), y)
    finally:
        plain.close()
        own.close()
        if own.other is not None:
            own.other.close()
