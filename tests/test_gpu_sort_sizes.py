"""The segment order at the sizes where the sort changes its form: one workgroup up to 4096 segments,
tiles of 256 .. 2048 that add up the histograms before them up to 524288, the scanned histograms above; exactly the
order numpy's lexsort gives (cell, window start, input index), for any number of segments of one cell."""
import numpy as np
import pytest
import torch

from helpers import segment_records

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 1025, 4095, 4096, 4097, 65536, 65537, 131073, 262145, 524288, 524289])
def test_segment_order(params4, lut, n):
    from larndsim_amd import synthetic
    from larndsim_amd.sim import Simulator

    p = params4.replace(number_pix_neighbors=0)
    base, f = synthetic.workload("c1")
    rng = np.random.default_rng(n)
    tr = base[rng.integers(0, len(base) if n % 2 else 7, n)].copy()  # even sizes: all in a few cells
    tr[:, f.index("z")] = rng.uniform(1.0, 29.0, n)
    tr[rng.random(n) < 0.01, f.index("eventID")] = -1  # dropped segments sort last
    print(f"[sort] {n}", flush=True)
    sim = Simulator(p, lut)
    st = sim.forward(p, tr, f)
    torch.cuda.synchronize()
    rec, keys, order = segment_records(sim, st)
    n_cells = st.n_events * 2 * 144 * 284
    k, o = keys.astype(np.int64), order.astype(np.int64)
    assert np.array_equal(np.sort(o), np.arange(n))
    assert (np.diff(k) >= 0).all()
    valid = k < n_cells
    S = np.clip(1950 - int(p.signal_length) - rec["k0"][valid].astype(np.int64), 0, 2002)
    assert np.array_equal(np.lexsort((o[valid], S, k[valid])), np.arange(valid.sum()))
    pids = st.out["pixel_ids"][: int(st.out["n_rows"].item())].cpu().numpy()
    assert (np.diff(pids) > 0).all()
