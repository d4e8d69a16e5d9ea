"""A row's float32 sum has a defined order, since a near tie at the threshold, and so a hit's tick, hangs on it:
the pairs of far and side cells by blocks of 64 to the waves in turn, the centre cell's segments one by one to the waves
in turn, each wave's in order, then the waves' partial rows in order.  With every segment in one pixel the terms
are the rows of events of one segment each, so the sum can be restated here, and equals the row bit for bit."""
import numpy as np
import pytest
import torch

from helpers import make_tracks, segment_records

pytestmark = pytest.mark.gpu


def _segments(p, n, seed):
    """n segments in the middle of one pixel (their diffusion bins stay inside it) at all depths, near the anode
    with windows that start before the first tick."""
    rng = np.random.default_rng(seed)
    b = np.asarray(p.tpc_borders)[0]
    at = lambda a, k: b[a, 0] + (k + 0.5) * p.pixel_pitch + rng.uniform(-0.01, 0.01, n)  # noqa: E731
    x, y, z = at(0, 30), at(1, 41), rng.uniform(min(b[2]) + 0.01, max(b[2]) - 0.01, n)
    return [dict(x=x[i], y=y[i], z=z[i], dE=rng.uniform(0.05, 2.0), dEdx=2.0, dx=0.2) for i in range(n)]


def _rows(sim, p, tr, f, n_events, px, py):
    st = sim.forward(p, tr, f, n_events=n_events)
    torch.cuda.synchronize()
    ids = st.out["pixel_ids"][: st.max_rows].cpu().numpy()
    nx, ny = int(p.n_pixels_x), int(p.n_pixels_y)
    at = np.nonzero((ids % nx == px) & (ids // nx % ny == py))[0]
    assert len(at) == n_events
    return st, st.out["wfs"][: st.max_rows].cpu().numpy()[at]


@pytest.mark.parametrize("a,b,n,waves", [(2, 0, 64, 4), (2, 0, 65, 4), (-4, 4, 700, 4), (3, -1, 300, 1), (-2, -3, 700, 8),
                                         (1, 0, 300, 4), (0, 0, 65, 4), (0, 0, 700, 4), (0, 0, 90, 2)])
def test_row_is_the_ordered_sum(params4, lut, a, b, n, waves):
    from larndsim_amd import sim as S

    p = params4
    # a segment without charge gives the row (a, b) pixels away
    bd = np.asarray(p.tpc_borders)[0]
    maker = dict(x=bd[0, 0] + (30 + a + 0.5) * p.pixel_pitch, y=bd[1, 0] + (41 + b + 0.5) * p.pixel_pitch, z=10.0, dE=0.0,
                 dEdx=2.0, dx=0.2)
    seg = _segments(p, n, 7 * n + waves)
    joint, f = make_tracks([maker] + seg)
    apart, _ = make_tracks([dict(s, eventID=e) for e in range(n) for s in (maker, seg[e])])
    sim = S.Simulator(p, lut)
    S.set_row_waves(waves)
    print(f"[row order] offset ({a}, {b}), {n} segments, {waves} waves", flush=True)
    try:
        st, row = _rows(sim, p, joint, f, 1, 30 + a, 41 + b)
        _, term = _rows(sim, p, apart, f, n, 30 + a, 41 + b)
    finally:
        S.set_row_waves(4)
    _, _, order = segment_records(sim, st)
    order = [int(i) for i in order if a == b == 0 or i > 0]  # (the maker shares the centre's cell)
    part = np.zeros((waves, row.shape[1]), np.float32)
    for k, i in enumerate(order):
        if i > 0:
            part[k % waves if a == b == 0 else k // 64 % waves] += term[i - 1]
    want = np.zeros(row.shape[1], np.float32)
    for w in range(waves):
        want += part[w]
    assert np.abs(want).max() > 0
    assert np.array_equal(row[0], want), f"{(row[0] != want).sum()} ticks differ"
