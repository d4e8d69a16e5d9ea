"""How exactly the waveform adjoint (k_rows_adj_dense) sums a window: it is linear in the cotangent, so the gradient of a
random cotangent on one row is compared with the same sum, in float64, over the gradients of single ticks, which need no
sum.  Tables and charges cancel out of that; what is left is the rounding of the sums.  They are float64 sums but for
the templates' differences, added three at a time in float32: a product's and two partial sums' roundings, 2^-24 (0.425
rms of a rounding) sqrt((1 + 2 + 3) / 3) = 0.60 2^-24 of the root of the summed squares of the terms, times the share that
the independent roundings of the cells' windows, much alike, have of their weighted sum.  The bound is 0.85 2^-24 times
that share, over 300 mixed cotangents, for every parameter, also where a window's terms cancel between the two ticks it is
split over or between cells (float32 sums of twelve terms leave 0.9 2^-24 without cancellation, and up to 40)."""
import numpy as np
import pytest
import torch

from helpers import make_tracks, segment_records

pytestmark = pytest.mark.gpu


def _cells_share(rec):
    """Root of the summed squares over the sum of the weights of a centred segment's merged cells."""
    def axis(u, w, nsb=10):
        cells = {}
        for k in range(5):
            c = (abs(2 * (u + k - 2) - nsb + 1) - 1) // 2
            cells[c] = cells.get(c, 0.0) + float(w[k])
        return np.array(list(cells.values()))

    W = np.outer(axis(rec["uxy"] & 0xffff, rec["wx"]), axis(rec["uxy"] >> 16, rec["wy"]))
    return np.sqrt((W ** 2).sum()) / W.sum()


# rows of a pixel that one segment reaches by its raw response, and of the segment's own pixel (diffusion bins)
@pytest.mark.parametrize("a,b,params", [(2, 0, (0, 1, 2, 3)), (-3, 4, (0, 1, 2, 3)), (0, 0, (0, 1, 2, 3, 5, 6))])
def test_rounding_of_the_window_sums(params4, lut, a, b, params):
    from larndsim_amd.sim import Simulator

    p = params4
    bd = np.asarray(p.tpc_borders)[0]
    at = lambda k, i: bd[k, 0] + (i + 0.5) * p.pixel_pitch  # noqa: E731
    tr, f = make_tracks([dict(x=at(0, 30) + 0.003, y=at(1, 41) - 0.002, z=12.0, dE=0.7, dEdx=2.0, dx=0.2),
                         dict(x=at(0, 30 + a), y=at(1, 41 + b), z=12.0, dE=0.0, dEdx=2.0, dx=0.2)])
    sim = Simulator(p, lut)
    st = sim.forward(p, tr, f, want_tape=True)
    ids = st.out["pixel_ids"][: st.max_rows].cpu().numpy()
    nx, ny = int(p.n_pixels_x), int(p.n_pixels_y)
    row = int(np.nonzero((ids % nx == 30 + a) & (ids // nx % ny == 41 + b))[0][0])
    ticks = np.nonzero(st.out["wfs"][row].cpu().numpy())[0]
    ticks = np.arange(max(ticks[0] - 2, 0), min(ticks[-1] + 3, sim.nout))
    zero = torch.zeros(st.max_rows, sim.H)
    print(f"[dense sums] offset ({a}, {b}), ticks {ticks[0]} to {ticks[-1]}", flush=True)

    def gradient(at, value):
        G = torch.zeros(st.max_rows, sim.nout)
        G[row, torch.as_tensor(at)] = torch.as_tensor(value, dtype=torch.float32)
        return sim.backward(st, zero, None, G).cpu().numpy()[list(params)]

    J = np.stack([gradient([o], [1.0]) for o in ticks])
    assert (np.abs(J).max(axis=0) > 0).all()
    rng = np.random.default_rng(3 + a)
    err = []
    for _ in range(300):
        G = rng.normal(size=len(ticks)).astype(np.float32)
        terms = G[:, None].astype(np.float64) * J
        err.append((gradient(ticks, G) - terms.sum(axis=0)) / np.sqrt((terms ** 2).sum(axis=0)))
    rms = np.sqrt(np.mean(np.square(err), axis=0))
    share = _cells_share(segment_records(sim, st)[0][0]) if a == b == 0 else 1.0
    print("[dense sums] rms error in 2^-24:", rms * 2 ** 24, "share", share, flush=True)
    assert (rms <= 0.85 * share * 2.0 ** -24).all()
