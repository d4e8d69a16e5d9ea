"""Segment records and boundary corrections made by one wave per 64 segments (many segments) and in parts on
several waves (few): the same arithmetic, so an event's waveforms are bit for bit those it has alone when
another event takes the launch over the line at 65536 segments, for every neighbourhood size."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nn", [0, 1, 2, 4])
def test_parts_equal_whole(params4, lut, nn):
    from larndsim_amd import synthetic
    from larndsim_amd.sim import Simulator

    p = params4.replace(number_pix_neighbors=nn)
    a, f = synthetic.workload("c1")
    a = a[:999].copy()
    ev = f.index("eventID")
    a[:, ev] = 0
    other = np.repeat(a[:1], 65536 - len(a) + 1, axis=0)  # one pixel of a second event
    other[:, ev] = 1
    other[:, f.index("dE")] *= 1e-3
    sim = Simulator(p, lut)
    print(f"[records] nn={nn}", flush=True)
    one = sim.forward(p, a, f)
    both = sim.forward(p, np.concatenate([a, other]), f)
    torch.cuda.synchronize()
    P = int(one.out["n_rows"].item())
    assert P > 10 and torch.equal(one.out["pixel_ids"][:P], both.out["pixel_ids"][:P])
    assert torch.equal(one.out["wfs"][:P], both.out["wfs"][:P])
