"""The kernel sums of two hit clouds check their shapes and devices before anything reaches the GPU."""
import pytest
import torch


@pytest.mark.parametrize("bad", ["coordinates", "weights", "events", "device"])
def test_shapes_are_checked(bad):
    from larndsim_amd import losses

    x, p, e = torch.zeros(4, 3).double(), torch.ones(4).double(), torch.zeros(4, dtype=torch.int64)
    y = torch.zeros(4, 2).double() if bad == "coordinates" else x
    q = p[:, None] if bad == "weights" else p
    f = e[:3] if bad == "events" else e
    if bad == "device":
        f = torch.zeros(4, dtype=torch.int64, device="meta")
    with pytest.raises(ValueError):
        losses._mmd_sums_hip(x, p, e, y, q, f, 1.0)
