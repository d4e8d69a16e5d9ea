"""The probabilistic readout evaluates once what ticks share (runs of equal cumulative charge, groups of
ticks with equal neighbours): rows that share nearly everything, nothing, and parts, at row lengths around
the 256-thread chunks and at the limits of rows and paths, against the same float64 oracle and to the same
bars as test_gpu_probfee.py and test_gpu_probfee_adjoint.py."""
import numpy as np
import pytest
import torch

from test_gpu_probfee import _compare
from test_gpu_probfee_adjoint import _check

pytestmark = pytest.mark.gpu


def _rows(kind, P, T, seed):
    """flat: pulses on zero; part: pulses and a pedestal on a third of the ticks; dense: on all."""
    rng = np.random.default_rng(seed)
    w = np.zeros((P, T), np.float32)
    for p in range(P):
        if kind != "flat":
            a = 0 if kind == "dense" else int(rng.integers(0, max(2 * T // 3, 1)))
            b = T if kind == "dense" else a + T // 3
            w[p, a:b] = rng.uniform(5, 60, size=b - a)
        for t in rng.choice(max(T - 12, 1), size=min(3, max(T - 12, 1)), replace=False):
            wd = int(min(rng.integers(2, 7), T - t))
            w[p, t:t + wd] += np.float32(rng.uniform(9000, 50000) / wd / 0.1)
    return w


@pytest.mark.parametrize("kind", ["flat", "part", "dense"])
@pytest.mark.parametrize("T,V", [(3, 1), (33, 20), (256, 20), (257, 1), (511, 32), (2048, 20)])
def test_forward(kind, T, V):
    from larndsim_amd import consts

    p = consts.default_params(RESET_NOISE_CHARGE=900.0, fee_paths_scaling=V, MAX_ADC_VALUES=3)
    assert _compare(p, _rows(kind, 4, T, 7 * T + V)) >= 4


# (dense rows of 2048 ticks leave too few rows without near ties to compare; test_gpu_probfee_adjoint.py
# has dense rows of 2000)
@pytest.mark.parametrize("T,kind", [(257, "part"), (512, "part"), (2048, "part"), (257, "dense"), (512, "dense")])
def test_adjoint(params4, kind, T):
    params = params4.replace(RESET_NOISE_CHARGE=900.0, MAX_ADC_VALUES=4)
    _check(params, _rows(kind, 4, T, T), 3)


def test_adjoint_of_flat_ticks():
    """Pulses on zero: moving the waveform on a flat stretch moves the outputs as differences say (the
    charge, which has no decision in it: d sum(charge) / d w in closed form over the row)."""
    from larndsim_amd import consts
    from larndsim_amd.fee import get_adc_values_average_noise_vmap

    p = consts.default_params(RESET_NOISE_CHARGE=900.0)
    T = 2000
    w = torch.from_numpy(_rows("flat", 3, T, 5)).cuda().requires_grad_(True)
    lp, q = get_adc_values_average_noise_vmap(p, w)
    run = (q != 0).any(dim=2)  # steps that ran
    q.sum().backward()
    # charge[t] = Q[sh(t)] + theta - (Q[t+1] + Q[t]) / 2 of each step that ran, Q the cumulative sum of w ts
    t = np.arange(T - 1)
    sh = np.minimum(t + p.adc_interval + 1, T - 1)
    dQ = np.zeros(T)
    np.add.at(dQ, sh, 1.0)
    np.add.at(dQ, t, -0.5)
    np.add.at(dQ, t + 1, -0.5)
    ref = np.cumsum(dQ[::-1])[::-1] * p.t_sampling
    for r in range(3):
        g = w.grad[r].double().cpu().numpy()
        n = int(run[r].sum())
        assert n >= 1
        np.testing.assert_allclose(g, n * ref, rtol=0, atol=1e-5 * n)
