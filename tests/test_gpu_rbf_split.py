"""The grid form of the event-blocked kernel sums where its workgroups' sharing of the candidates has edges:
one query up to a few around the 64 of a workgroup, fewer candidates than waves, several events within one
workgroup, and queries so scattered that a workgroup walks more than 512 columns.  Against the sums over every pair in
float64 on the CPU: float32 distances of coordinates up to 100 cm with d^2 / (2 sigma^2) < 106 give a kernel
value to ~106 * 4 * 2^-24 + the exponential's rounding = 3e-5 of itself at the far end, where it is 1e-46 of the
near ones; relative to the sum of |terms| the rounding of coordinates close to each other (2^-24) and of runs
of 32 terms (2e-6) leaves 4e-6.  Queries are placed next to a candidate so that near terms exist."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,events,sigma", [(1, 1, 1, 1.0), (63, 7, 1, 1.0), (64, 8, 1, 1.0), (65, 9, 1, 1.0),
                                                (130, 3, 40, 1.0), (129, 513, 3, 0.5), (70, 2000, 1, 0.5),
                                                (70, 2000, 1, 8.0)])
def test_grid_sums_at_the_edges(nx, ny, events, sigma):
    from larndsim_amd import losses

    g = np.random.default_rng(nx + ny)
    y = torch.tensor(g.integers(-400, 400, (ny, 3)) * 0.25, dtype=torch.float32)  # (exact distances)
    ey = torch.tensor(g.integers(0, events, ny))
    k = torch.tensor(g.integers(0, ny, nx))
    x = y[k] + torch.tensor(g.integers(-2, 3, (nx, 3)) * 0.25, dtype=torch.float32)
    ex = torch.where(torch.tensor(g.random(nx) < 0.9), ey[k], torch.tensor(events))  # (some without any candidate)
    c = torch.tensor(g.normal(size=(ny, 4)), dtype=torch.float32).double()
    print(f"[rbf-split] nx {nx} ny {ny} events {events} sigma {sigma}", flush=True)
    got = losses._block_sums(x.cuda(), ex.cuda(), y.cuda(), ey.cuda(), c.cuda(), sigma).cpu()
    d2 = ((x.double()[:, None] - y.double()[None]) ** 2).sum(-1) / (2 * sigma * sigma)
    K = torch.exp(-d2) * (ex[:, None] == ey[None])
    want, scale = K @ c, K @ c.abs()
    some = scale[:, 0] > 0
    assert some.any()
    err = ((got - want).abs()[some] / scale[some]).max().item()
    print(f"[rbf-split] error / sum|terms| {err:.2e}", flush=True)
    assert err < 4e-6
    assert torch.equal(got[~some], torch.zeros_like(got[~some]))
