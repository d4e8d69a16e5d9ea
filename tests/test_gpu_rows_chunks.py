"""The waveform kernel's time chunks: window lengths at the edges of the 64-tick chunks, windows that
start before the first tick, rows of one and of several batches of pairs, and pairs with a non-finite
charge, against the float64 oracle (1e-5 of each row's peak, the bar of the other waveform tests: a sum of
n float32 terms is off by about sqrt(n) 2^-24 of its largest partial sum, 4e-6 for the 4000 pairs here)."""
import numpy as np
import pytest
import torch

from helpers import compare_forward, make_tracks
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _event(p, n, seed, spread):
    """n segments within `spread` cm of a pixel corner, all drift depths: near the anode the windows start
    before the first output tick."""
    rng = np.random.default_rng(seed)
    b = np.asarray(p.tpc_borders)[0]
    c = (b[0, 0] + 30 * p.pixel_pitch, b[1, 0] + 41 * p.pixel_pitch)
    z = rng.uniform(min(b[2]) + 0.01, max(b[2]) - 0.01, n)
    return make_tracks([dict(x=c[0] + rng.uniform(-spread, spread), y=c[1] + rng.uniform(-spread, spread), z=z[i], dE=0.4,
                             dEdx=2.0, dx=0.2) for i in range(n)])


@pytest.mark.parametrize("L", [1, 63, 64, 65, 127, 128, 129, 187])
def test_window_lengths(params4, lut, L):
    from larndsim_amd.sim import Simulator

    p = params4.replace(signal_length=L)
    tr, f = _event(p, 150, L, 0.9)
    compare_forward(Simulator(p, lut), p, lut, tr, f, tag=f"L{L}")


@pytest.mark.parametrize("n,spread,waves", [(1, 0.1, 4), (65, 0.2, 4), (1600, 0.15, 4), (4000, 0.4, 4), (4000, 0.4, 1), (4000, 0.4, 8)])
def test_pairs_per_row(params4, lut, n, spread, waves):
    from larndsim_amd import sim as S

    tr, f = _event(params4, n, n, spread)
    S.set_row_waves(waves)
    try:
        compare_forward(S.Simulator(params4, lut), params4, lut, tr, f, tag=f"n{n} w{waves}")
    finally:
        S.set_row_waves(4)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_non_finite_charge(params4, lut, bad):
    """A segment with a non-finite energy spoils the ticks its windows reach and no others: up to the first
    of them, and on rows it does not reach, the waveforms are those of the event without it."""
    from larndsim_amd.sim import Simulator

    sim = Simulator(params4, lut)
    tr, f = _event(params4, 300, 5, 3.0)
    i = int(np.argmin(np.abs(tr[:, f.index("z")] - 15.0)))
    spoiled, without = tr.copy(), tr.copy()
    spoiled[i, f.index("dE")] = bad
    without[i, f.index("dE")] = 0.0
    a = sim.forward(params4, spoiled, f)
    b = sim.forward(params4, without, f)
    torch.cuda.synchronize()
    wa, wb = (s.out["wfs"][: s.max_rows].cpu().numpy() for s in (a, b))
    assert np.array_equal(a.out["pixel_ids"][: a.max_rows].cpu().numpy(), b.out["pixel_ids"][: b.max_rows].cpu().numpy())
    q = O.segment_quantities(params4, tr[i:i + 1], f)
    S = lut.shape[2] - int(params4.signal_length) - int(np.floor(q["tau"][0]))
    hit = ~np.isfinite(wa).all(axis=1)
    assert hit.any()
    peak = np.abs(wb).max(axis=1, keepdims=True) + 1e-30
    near = np.abs(wa[:, : S - 2] - wb[:, : S - 2]) / peak
    assert near.max() < 1e-5
    assert (np.abs(wa[~hit] - wb[~hit]) / peak[~hit]).max() < 1e-5
    ok = np.abs(wa[hit][:, S + 187:] - wb[hit][:, S + 187:]) / peak[hit]
    assert ok.max() < 1e-5
    ticks = a.out["ticks"][: a.max_rows].cpu().numpy()[hit]
    assert ((ticks < S + 187) | (ticks >= sim.nout - 3)).all()  # no hit after the charge has become NaN
