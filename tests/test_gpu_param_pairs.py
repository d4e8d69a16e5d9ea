"""The closed form of the current's exponentially modified Gaussian and the pairs' hand-over within a wave
(k_param_rows), against the float64 oracle (oracle/param.py): a pixel with 1 pair up to several full
hand-overs of 4 waves x 64 pairs, and longitudinal spreads from far narrower than a tick to far wider than the
5 us window, as well as none at all.  Bound 1e-6 of a row's peak: the float32 result rounds at 6e-8 and the sums are
float64; rows that overflow in the oracle overflow here."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pairs,long_diff", [(1, 1.0), (3, 1.0), (4, 1.0), (255, 1.0), (256, 1.0), (257, 1.0), (700, 1.0),
                                             (300, 1e-12), (300, 30.0), (300, 1e3), (300, 0.0)])
def test_pairs_of_one_pixel(params4, c1, pairs, long_diff):
    from larndsim_amd import param as GP
    from oracle import param as PA

    tr, f = c1
    tr = np.repeat(np.ascontiguousarray(tr[:1]), pairs, axis=0)
    rng = np.random.default_rng(pairs)
    for c in "xyz":  # within a pixel or so of each other, over a few drift ticks
        k = f.index(c)
        tr[:, k] += rng.normal(scale=0.3 if c == "z" else 0.05, size=pairs).astype(tr.dtype)
    p = params4.replace(mc_diff=True, number_pix_neighbors=0, diffusion_in_current_sim=True,
                        long_diff=params4.long_diff * long_diff)
    normals = np.zeros((pairs, 3), np.float32)
    print(f"[param pairs] {pairs} long_diff x {long_diff}", flush=True)
    e = GP.electrons(p, torch.from_numpy(tr).cuda(), f, normals=torch.from_numpy(normals).cuda())
    wfs, U = GP.waveforms(p, e)
    with np.errstate(all="ignore"):
        o = PA.simulate_parametrized(p, tr, f, normals=normals.astype(np.float64))
    U = U.cpu().numpy()
    assert np.array_equal(U, o["unique_pixels"])
    valid = U >= 0
    assert valid.any()
    g, w = wfs.cpu().numpy().astype(np.float64)[valid], o["wfs"][:, 1:][valid]
    nan = np.isnan(w).any(axis=1)
    assert np.array_equal(np.isnan(g).any(axis=1), nan)
    assert nan.all() == (long_diff == 1e3)  # (there every row overflows)
    g, w = g[~nan], w[~nan]
    if len(w):
        err = (np.abs(g - w) / (np.abs(w).max(axis=1, keepdims=True) + 1e-30)).max()
        print(f"[param pairs] error / row peak {err:.2e}", flush=True)
        assert err < 1e-6
