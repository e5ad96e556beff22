"""State that differentiated propagations share: kernel spectra by grid and
distance, CZT tables by geometry.  What may be shared, and what may not.
"""
import numpy as np
import pytest
import torch

from oracle import xlumina_ref as R
from tests.conftest import rel_l2
from xlumina_amd import _native as N
from xlumina_amd import autograd as AG

CPU = torch.device("cpu")


def _rs_config(x, y=None, z=40.0):
    return AG.RSConfig(x, x if y is None else y, z, 0.65, N.XL_EZ_NONE, 1)


def test_spectra_key_follows_a_grid_changed_in_place():
    x, y = (torch.linspace(-8.0, 8.0, 16, dtype=torch.float64) for _ in range(2))
    cfg = _rs_config(x, y)
    key = AG._spectra_key(cfg, None, 16, 1, CPU)[0]
    assert AG._spectra_key(cfg, None, 16, 1, CPU)[0] == key
    for grid in (x, y):
        grid.mul_(2)
        changed = AG._spectra_key(cfg, None, 16, 1, CPU)[0]
        assert changed != key
        key = changed


def test_spectra_of_untracked_grids_are_not_shared():
    with torch.inference_mode():
        x = torch.linspace(-8.0, 8.0, 16, dtype=torch.float64)
    assert AG._spectra_key(_rs_config(x), None, 16, 1, CPU)[0] is None


@pytest.mark.gpu
@pytest.mark.parametrize("axis", ["x", "y"])
def test_propagation_after_a_device_grid_changed_in_place(cuda_dev, axis):
    """A device grid stretched between two differentiated calls, the first
    one's output alive: the second propagates over the new grid (oracle,
    relative L2 <= 1e-5, the FP32 paths' bar)."""
    n, z, wl = 48, 900.0, 0.65
    rng = np.random.default_rng(3)
    f = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    src = torch.tensor(f.astype(np.complex64), device=cuda_dev)[None].requires_grad_(True)
    g = {k: torch.linspace(-100.0, 100.0, n, dtype=torch.float64, device=cuda_dev) for k in "xy"}
    first = AG.rs(src, g["x"], g["y"], z, wl)
    g[axis].mul_(2)
    second = AG.rs(src, g["x"], g["y"], z, wl)
    x, y = (g[k].cpu().numpy() for k in "xy")
    assert rel_l2(second.detach()[0].cpu().numpy(), R.rs_propagation(f, x, y, wl, z)[0]) < 1e-5
    assert first.requires_grad
