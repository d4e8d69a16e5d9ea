"""Rows handed to workgroups by runs of 16 over 8 XCDs: every row is computed once, and the places past the
last row count no hits and add no gradient, for row counts around the run and around a round of runs and for
buffers with room for more rows than there are.  Row by row the results are those of an exact buffer, bit for bit."""
import numpy as np
import pytest
import torch

from helpers import make_tracks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 15, 16, 17, 127, 128, 129, 300])
def test_rows_and_room(params4, lut, P):
    from larndsim_amd.sim import Simulator

    p = params4
    b = np.asarray(p.tpc_borders)[0]
    tr, f = make_tracks([dict(x=b[0, 0] + (20 + i % 20 + 0.5) * p.pixel_pitch, y=b[1, 0] + (20 + i // 20 + 0.5) * p.pixel_pitch,
                              z=2.0 + 0.08 * i, dE=2.0, dEdx=2.0, dx=0.2) for i in range(P)])
    sim = Simulator(p, lut)
    g = torch.Generator().manual_seed(P)
    print(f"[runs] {P} rows", flush=True)
    exact = sim.forward(p, tr, f, n_events=1, want_tape=True)
    assert exact.max_rows == P
    G = torch.randn(P, sim.nout, generator=g)
    d_adc = torch.randn(P, sim.H, generator=g)
    n_hits = int(exact.out["n_hits"].item())
    assert n_hits >= P // 2
    grads = [sim.backward(exact, d_adc, None, w) for w in (None, G)]
    for room in (1, 130):
        # (the library takes no more rows than segments: repeat dropped segments to make room)
        pad = np.repeat(tr[:1], room, axis=0)
        pad[:, f.index("eventID")] = -1
        st = sim.forward(p, np.concatenate([tr, pad]), f, n_events=1, want_tape=True, max_rows=P + room)
        assert int(st.out["n_rows"].item()) == P and int(st.out["n_hits"].item()) == n_hits
        assert torch.equal(st.out["wfs"][:P], exact.out["wfs"][:P])
        assert torch.equal(st.out["hit_tick"][:n_hits], exact.out["hit_tick"][:n_hits])
        da = torch.cat([d_adc, torch.ones(room, sim.H)])
        for want, w in zip(grads, (None, torch.cat([G, torch.ones(room, sim.nout)]))):
            got = sim.backward(st, da, None, w)
            assert torch.allclose(got, want, rtol=1e-12, atol=0.0), (got, want)
