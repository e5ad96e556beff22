"""Plane-factor tables of batched RS-mode CZTs: built beside the axis tables
where both axes have one transform length, in a launch of their own otherwise.
Each member of a batch of four (tables) against its own call (no tables), on
rectangular planes, both directions, at table sizes around the launch's blocks.
Both evaluate the factors by the same float64 expressions and round them once,
so 1e-6 in relative L2 leaves room for the order of the float32 products only.
"""
import numpy as np
import pytest
import torch

from xlumina_amd import ops

pytestmark = pytest.mark.gpu


# (nx, ny, mx, my): one length on both axes (64, 128, 512, 2048), then two lengths
SIZES = [(2, 2, 2, 2), (33, 29, 20, 31), (130, 131, 90, 77), (700, 701, 500, 333), (250, 40, 99, 20), (100, 600, 60, 300)]


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("nx,ny,mx,my", SIZES)
def test_batch_with_tables_equals_alone(nx, ny, mx, my, adjoint):
    gen = torch.Generator(device="cuda").manual_seed(nx + 4096 * ny)
    x, y = np.linspace(-1.1 * nx, 0.9 * nx, nx), np.linspace(-ny, 1.2 * ny, ny)
    xo, yo = np.linspace(-0.3 * nx, 0.35 * nx, mx), np.linspace(-0.2 * ny, 0.3 * ny, my)
    g = ops.czt_geometry(x, y, xo, yo, 3e4, 0.635)
    plane = (my, mx) if adjoint else (ny, nx)
    src = torch.randn((4, 1, *plane), generator=gen, device="cuda", dtype=torch.complex64)
    out = ops.czt(src, g, adjoint=adjoint, batch=4)
    assert out.shape == (4, 1, *((ny, nx) if adjoint else (my, mx)))
    for b in range(4):
        alone = ops.czt(src[b], g, adjoint=adjoint, form="bluestein").to(torch.complex128)
        assert float((out[b].to(torch.complex128) - alone).norm()) <= 1e-6 * float(alone.norm())
