"""Rows written where the reference's layout has them (Simulator.forward_reference_rows) against the plain
rows laid out afterwards (reference_rows), bit for bit: ordinary events, padding segments (negative pixel
ids), segments off the pixel plane, an event without any row and one without any segment."""
import numpy as np
import pytest
import torch

from helpers import mixed_event

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["c1", "mixed", "padding", "none"])
def test_rows_in_place(params4, lut, kind):
    from larndsim_amd import sim as S
    from larndsim_amd import synthetic

    if kind == "mixed":
        tr, f = mixed_event(params4)
    else:
        tr, f = synthetic.workload("c1")
        tr = tr[:300].copy()
        if kind == "padding":
            tr[:] = 0.0
            tr[:, f.index("eventID")] = -1
        if kind == "none":
            tr = tr[:0]
    sim = S.Simulator(params4, lut)
    print(f"[rows] {kind}", flush=True)
    st0 = sim.forward(params4, tr, f, n_events=1)
    neg, n_neg = sim.negative_rows(params4, st0.seg)
    S.size_history_dict.clear()
    want = S.reference_rows(st0.out["wfs"][: st0.max_rows], st0.out["pixel_ids"][: st0.max_rows], neg, n_neg)
    S.size_history_dict.clear()
    st, wfs, ids = sim.forward_reference_rows(params4, tr, f, n_events=1)
    assert st.max_rows == st0.max_rows and (st.max_rows == 0) == (kind in ("padding", "none"))
    assert (int(n_neg.item()) > 0) == (kind in ("mixed", "padding"))
    assert torch.equal(ids, want[1]) and torch.equal(wfs, want[0])
    a, b = S.hits_dict(st.out), S.hits_dict(st0.out)
    assert all(torch.equal(a[k], b[k]) for k in a)
    assert int(st.out["status"].item()) == int(st0.out["status"].item())
