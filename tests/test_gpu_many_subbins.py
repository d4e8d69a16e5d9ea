"""More than 256 sub-bins a pixel: sub-bin positions that need nine bits on both axes reach the waveform kernel and both
adjoints whole.  A response table of independent random windows (a wrong bin is a wrong window), segments all over
a few pixels and at their edges, close to the cathode, where the short table's time axis has their arrival; against the
float64 oracle and its autograd at the bars of the other forward and adjoint tests (1e-5 of a row's peak, 1e-3)."""
import numpy as np
import pytest
import torch

from helpers import compare_forward, make_tracks

pytestmark = pytest.mark.gpu

NSB, NT, L = 260, 64, 40


@pytest.fixture(scope="module")
def event(params4):
    p = params4.replace(nb_sampling_bins_per_pixel=NSB, number_pix_neighbors=1, signal_length=L, long_diff_extent=8,
                        long_diff_template=np.linspace(0.001, 10, 4).astype(np.float32))
    rng = np.random.default_rng(9)
    lut = rng.normal(scale=0.05, size=(NSB + NSB // 2, NSB + NSB // 2, NT)).astype(np.float32)
    lut[: NSB // 2, : NSB // 2] += 0.2  # charge is collected inside the pixel
    b = np.asarray(p.tpc_borders)[0]
    n = 160
    w = p.pixel_pitch / NSB
    at = rng.uniform(0, 3 * NSB, size=(n, 2))
    edge = rng.random((n, 2)) < 0.3  # within three sub-bins of a pixel's edge
    at = np.where(edge, np.clip(np.round(at / NSB) * NSB + rng.uniform(-3, 3, size=(n, 2)), 0.1, 3 * NSB - 0.1), at)
    assert (np.floor(at % NSB) > 255).any(axis=1).sum() > 5
    z = b[2, 1] + np.sign(b[2, 0] - b[2, 1]) * rng.uniform(0.05, 0.9, n)
    tr, f = make_tracks([dict(x=b[0, 0] + 30 * p.pixel_pitch + at[i, 0] * w, y=b[1, 0] + 41 * p.pixel_pitch + at[i, 1] * w,
                              z=z[i], dE=1.0, dEdx=2.0, dx=0.2) for i in range(n)])
    return p, lut, tr, f


def test_forward(event):
    from larndsim_amd.sim import Simulator

    p, lut, tr, f = event
    st, ref = compare_forward(Simulator(p, lut), p, lut, tr, f, tag="260 sub-bins")
    assert st.max_rows == 9 and (ref["grid"]["ticks"] < 1997).any()


@pytest.mark.parametrize("waveforms", [False, True])
def test_adjoint(event, waveforms):
    from larndsim_amd.sim import Simulator
    from oracle import ad_oracle as A

    p, lut, tr, f = event
    fz = A.Frozen(p, lut, tr, f)
    sim = Simulator(p, lut)
    print(f"[260 sub-bins] adjoint, waveforms {waveforms}", flush=True)
    st = sim.forward(p, tr, f, want_tape=True)
    vr = fz.valid_rows
    assert st.max_rows == int(vr.sum())
    rng = np.random.default_rng(3)
    hits = fz.ticks[vr] < 1997
    d_adc = (rng.normal(size=hits.shape) * hits).astype(np.float32)
    G = rng.uniform(0.5, 1.5, size=(st.max_rows, sim.nout)).astype(np.float32) if waveforms else None
    th = fz.theta0().requires_grad_(True)
    adc, _, wfs = fz.forward(th)
    loss = (torch.as_tensor(d_adc.astype(np.float64)) * adc[torch.as_tensor(vr)]).sum()
    if waveforms:
        loss = loss + (torch.as_tensor(G.astype(np.float64)) * wfs[torch.as_tensor(vr)]).sum()
    loss.backward()
    want = th.grad.numpy()
    got = sim.backward(st, torch.from_numpy(d_adc), None, None if G is None else torch.from_numpy(G)).cpu().numpy()
    print("got ", got, "\nwant", want, flush=True)
    on = np.abs(want) > 0
    assert on.sum() >= 4
    assert (np.abs(got - want)[on] <= 1e-3 * np.abs(want)[on]).all()
