"""lsim_rbf_mmd_sums (bounds, grid, sort and both kernel sums of two hit clouds) against the sums over every pair
in float64: empty and single-point clouds, points all in one place (cells of no extent), negative event numbers,
events on one side only, sorts of one workgroup and of many.  Coordinates are multiples of 1/4 cm, so distances are
exact and the bound is that of the grid form: float32 runs of 32 terms (2e-6), products and exponential, 4e-6
of the sum of |terms|."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,events,spread,sigma", [(1, 0, 1, 10, 1.0), (0, 5, 1, 10, 1.0), (1, 1, 1, 10, 1.0),
                                                       (70, 64, 1, 0, 1.0), (300, 900, 4, 200, 0.5),
                                                       (3000, 2500, 2, 400, 1.0), (900, 3300, 3, 100, 4.0)])
def test_sums_of_two_clouds(nx, ny, events, spread, sigma):
    from larndsim_amd import losses

    g = np.random.default_rng(nx + ny)
    pos = lambda n: torch.tensor(g.integers(-spread, spread + 1, (n, 3)) * 0.25)  # noqa: E731
    x, y = pos(nx), pos(ny)
    px, py = (torch.tensor(g.uniform(0.5, 2.0, n)).float().double() for n in (nx, ny))
    ex = torch.tensor(g.integers(-1, events, nx))
    ey = torch.tensor(g.integers(0, events + 1, ny))
    print(f"[mmd] {nx} x {ny} events {events} sigma {sigma}", flush=True)
    got = losses._mmd_sums_hip(x.cuda(), px.cuda(), ex.cuda(), y.cuda(), py.cuda(), ey.cuda(), sigma)
    for out, b, pb, eb in zip(got, (x, y), (px, py), (ex, ey)):
        out = out.cpu()
        c = torch.cat([pb[:, None], pb[:, None] * b], dim=1)
        K = torch.exp(-((x[:, None] - b[None]) ** 2).sum(-1) / (2 * sigma * sigma)) * (ex[:, None] == eb[None])
        want, scale = K @ c, K @ c.abs()
        assert out.shape == want.shape
        if out.numel():
            # (sums of terms below 1e-25 are compared as zero)
            err = ((out - want).abs() / (scale + 1e-25)).max().item()
            print(f"[mmd] error / sum|terms| {err:.2e}", flush=True)
            assert err < 4e-6
