"""The fused generation's members per workgroup (4 up to 512 members, 8 up to 1,024, 16 beyond)
at the edges of those ranges and with a last workgroup that is partly empty: populations
bit-identical to the layered form's."""
import numpy as np
import pytest

from mcluminescence_amd import fit as F
from mcluminescence_amd import fit_bench
from mcluminescence_amd import surrogate as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def net(gpu_ctx):
    n = S.Network.load(gpu_ctx, fit_bench.MODEL, max_batch=4096)
    yield n
    n.close()


@pytest.mark.parametrize("pop", [4, 5, 33, 511, 512, 513, 519, 1023, 1025, 1041, 4096])
@pytest.mark.parametrize("dim", [5, 1])
def test_members_per_workgroup(net, pop, dim):
    import torch
    print(f"DE groups pop={pop} dim={dim}", flush=True)
    target = np.exp(-0.5 * ((np.arange(256) - 110.0) / 25.0) ** 2).astype(np.float32) * 40.0
    res = []
    for layered in (False, True):
        de = F.NetworkDE(net, target, 1.0e4, [0.1] * (6 - dim), dim, pop, seed=9, layered=layered)
        try:
            de.run(9)
            x, f = de.population()
            res.append((x.clone(), f.clone(), de.best()))
        finally:
            de.close()
    (xa, fa, ba), (xb, fb, bb) = res
    assert torch.equal(xa, xb) and torch.equal(fa, fb)
    np.testing.assert_array_equal(ba[0], bb[0])
    assert ba[1] == bb[1]
