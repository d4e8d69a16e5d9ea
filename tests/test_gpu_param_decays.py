"""Pairs whose current has a decay constant near zero, where the tails' exponentials leave the float64 range
(k_param_rows), tick by tick against the float64 oracle (oracle/param.py): one electron to a row, its distance
from the row's pixel such that the decay runs through zero, longitudinal spreads of 0.1 to 0.25 us.  A tail whose
normaliser overflows is zero where its own values are finite and NaN or infinite where they are not, and only there.
The oracle takes the C library's erfc here: SciPy's is 0 where the value is denormal, which makes NaN (infinity times
zero) of what is infinite.  Bound as for the other pairs: 1e-6 of the row's peak (float32 results of float64 sums), for
the rows without a denormal erfc, whose few bits the infinities and NaNs alone are checked of."""
import math

import numpy as np
import pytest
import torch

from helpers import make_tracks

pytestmark = pytest.mark.gpu


def _event(p, lo, hi, seed):
    """Electrons every 4 pixels, each with the decay constant c of detsim_jax.py:587 in [lo, hi] towards the next
    pixel in x, at random depths."""
    from oracle import param as PA

    rng = np.random.default_rng(seed)
    b = np.asarray(p.tpc_borders)[0]
    rows = []
    for px in range(2, int(p.n_pixels_x) - 2, 4):
        for py in range(2, int(p.n_pixels_y) - 2, 4):
            y = rng.uniform(0.0, 0.1)
            c0, cx, cy, cxy, cxx, cyy = PA.C_PARAMS
            k = c0 + cy * y + cyy * y * y - rng.uniform(lo, hi)
            q = cx + cxy * y
            x = (-q - np.sqrt(q * q - 4 * cxx * k)) / (2 * cxx)
            rows.append(dict(x=b[0, 0] + (px + 1.5) * p.pixel_pitch - x, y=b[1, 0] + (py + 0.5) * p.pixel_pitch + y,
                             z=rng.uniform(min(b[2]) + 1.0, max(b[2]) - 8.0), dE=0.5, dEdx=2.0, dx=0.2))
    return make_tracks(rows)


@pytest.mark.parametrize("lo,hi,n", [(0.003, 0.007, 1), (-0.02, 0.02, 1), (-1e-7, 1e-7, 1), (0.0, 0.05, 4)])
def test_decays_through_zero(params4, lo, hi, n, monkeypatch):
    from larndsim_amd import param as GP
    from oracle import param as PA

    tiny = []
    c_erfc = np.vectorize(math.erfc, otypes=[float])

    def erfc(x):
        v = c_erfc(x)
        tiny.append(((v > 0) & (v < 1e-300)).any(axis=-1))
        return v

    monkeypatch.setattr(PA, "erfc", erfc)
    p = params4.replace(mc_diff=True, number_pix_neighbors=n, diffusion_in_current_sim=True)
    tr, f = _event(p, lo, hi, int(1e6 * hi) + n)
    normals = np.zeros((len(tr), 3), np.float32)
    print(f"[param decays] {len(tr)} electrons, decays {lo} to {hi}, {n} neighbours", flush=True)
    e = GP.electrons(p, torch.from_numpy(tr).cuda(), f, normals=torch.from_numpy(normals).cuda())
    wfs, U = GP.waveforms(p, e)
    with np.errstate(all="ignore"):
        o = PA.simulate_parametrized(p, tr, f, normals=normals.astype(np.float64))
        w = o["wfs"][:, 1:].astype(np.float32)
    U = U.cpu().numpy()
    assert np.array_equal(U, o["unique_pixels"])
    valid = U >= 0
    coarse = np.isin(U, o["pair_pids"][np.any(tiny, axis=0)])[valid]
    g, w = wfs.cpu().numpy()[valid], w[valid]
    bad = np.isnan(w)
    print(f"[param decays] rows with NaN {bad.any(axis=1).sum()}, fewer than ten ticks of it "
          f"{(bad.any(axis=1) & (bad.sum(axis=1) < 10)).sum()}", flush=True)
    assert np.array_equal(np.isnan(g), bad)
    assert np.array_equal(np.isinf(g), np.isinf(w))
    fin = np.isfinite(w) & ~coarse[:, None]
    assert fin.any(axis=1).mean() > 0.8
    peak = np.where(fin, np.abs(w), 0.0).max(axis=1, keepdims=True) + 1e-30
    err = (np.where(fin, np.abs(g.astype(np.float64) - w), 0.0) / peak).max()
    print(f"[param decays] error / row peak {err:.2e}", flush=True)
    assert err < 1e-6
