"""The lab kernel at the edges of its rows and slots, bit-exact against the CPU replay: electron
counts around a row of 64 and around the 8 rows whose channel draws are kept, a cluster that
grows from empty through all of them, enough pairs that the hole slots are packed again, and
each loop option with the draws it adds."""
import numpy as np
import pytest

from mcluminescence_amd._abi import RunParams
from oracle import orc

pytestmark = pytest.mark.gpu

EXACT, SHARED, FIRST, RETRAP = 1, 2, 4, 8


def lab_run(n, T, start=0.0, D=0.092, retrap=0.5, sims=2):
    return RunParams.make(alpha=9e9, b=1e12, s=1e13, E_cb=1.8, E_loc_1=1.4, E_loc_2=1.42, D0=400.35,
                          Retrap=retrap, k_b=8.617333262e-5, D=D, rho_prime=1e-4, holes=float(n),
                          boundary_factor=1.2, N_e=float(n), e_ratio_start=start, T_start=T,
                          T_rate=-0.01, dt=1.0, n_steps=1, sims=sims)


def check(ctx, run, obs, options):
    ratio, status, stats = ctx.run_lab([run], [obs], options=options)
    ref, rstatus = orc.run_lab([run], [obs], options=options, threads=8)
    np.testing.assert_array_equal(status, rstatus)
    np.testing.assert_array_equal(ratio, ref)
    return stats


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 511, 513, 577])
@pytest.mark.parametrize("options", [0, EXACT, SHARED | FIRST | RETRAP])
def test_rows(gpu_ctx, n, options):
    print(f"lab rows n={n} options={options}", flush=True)
    check(gpu_ctx, lab_run(n, 150.0), [10.0, 500.0, 500.0, 4000.0], options)
    check(gpu_ctx, lab_run(n, 330.0, start=1.0, D=0.0), [0.0, 5.0, 400.0], options)


@pytest.mark.parametrize("options", [0, EXACT, RETRAP | EXACT, SHARED])
def test_slots_packed_again(gpu_ctx, options):
    # 20 electrons: 64 + 2 x 20 hole slots beyond the first ones, and several hundred pairs
    stats = check(gpu_ctx, lab_run(20, 330.0, D=20.0), [100.0, 3000.0], options)
    assert stats.recombinations > 400
