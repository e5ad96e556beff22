"""The forms that a pass is launched in, on both sides of the lines that choose
them: where the row-transformed RS kernel lies, rows with their components side
by side or one after the other, staged and direct CZT columns, and the row
blocks of the longest CZT rows.

Tolerances: the two sides of the first test run the same kernels on the same
numbers (equal bits).  Elsewhere two forms of one transform are each within
1e-6 of float64, so 2e-6 apart at most; the float64 oracle and the adjoint
identity are held to 1e-5, the FP32 paths' bar.
"""
import numpy as np
import pytest
import torch

from oracle import xlumina_ref as R
from tests.conftest import rel_l2
from xlumina_amd import _native as N
from xlumina_amd import ops
from xlumina_amd.ops import MaskSpec

pytestmark = pytest.mark.gpu


def gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def cplx(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.complex64)


def uni(g, *shape):
    return 6 * torch.rand(shape, generator=g, device="cuda")


def near(a, b, tol):
    a, b = a.to(torch.complex128), b.to(torch.complex128)
    assert a.shape == b.shape and float((a - b).norm()) <= tol * float(b.norm()), float((a - b).norm() / b.norm())


def adjoint_identity(f, af, g, hg):
    f, af, g, hg = (t.to(torch.complex128) for t in (f, af, g, hg))
    assert abs(complex((g.conj() * af).sum() - (hg.conj() * f).sum())) <= 1e-5 * float(g.norm() * af.norm())


# a call that keeps its kernel spectrum has room for all of the row-transformed kernel beside it; a plain call for all,
# seven eighths (2n - 1 close to a power of two) or none of it (up to 128 points)
@pytest.mark.parametrize("n", [2, 13, 14, 16, 17, 32, 57, 64, 65, 100, 126, 128, 200, 250, 256, 257, 512, 1003, 1008,
                               1024, 1537, 2047, 2048])
def test_kernel_rows_in_either_place(cuda_dev, n):
    g = gen(n)
    x = np.linspace(-1.2 * n, 1.2 * n, n)
    src = cplx(g, 2, n, n)
    hh = torch.empty(ops.rs_hhat_bytes(n), dtype=torch.uint8, device=cuda_dev)
    for kw in (dict(ez_mode=N.XL_EZ_VRS, nin=2, masks=[MaskSpec(N.XL_MASK_SSLM, uni(g, n, n), uni(g, n, n))]),
               dict(nin=1)):
        a = ops.rs_propagate(src, x, x, 30.0 * n, 0.65, **kw)
        b = ops.rs_propagate(src, x, x, 30.0 * n, 0.65, hhat=hh, hhat_mode=1, **kw)
        assert torch.equal(a, b)


@pytest.mark.parametrize("n", [2, 3, 29, 31, 63, 66, 127, 130, 255])
def test_rows_of_two_components(cuda_dev, n):
    rng = np.random.default_rng(n)
    x, y = R.space(3.0 * n, n)
    e = rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))
    p = rng.uniform(-np.pi, np.pi, (2, n, n)).astype(np.float32)
    masks = [MaskSpec(N.XL_MASK_SSLM, *(torch.tensor(v, device=cuda_dev) for v in p))]
    out = ops.rs_propagate(torch.tensor(e.astype(np.complex64), device=cuda_dev), x, y, 40.0 * n, 0.65, masks=masks)
    for i in range(2):
        ref = R.rs_propagation(e[i] * np.exp(1j * p[i].astype(np.float64)), x, y, 0.65, 40.0 * n)[0]
        assert rel_l2(out[i].cpu().numpy(), ref) < 1e-5


# members whose rows together stay within or exceed 2048
@pytest.mark.parametrize("n,batch", [(64, 40), (128, 17), (250, 8), (250, 9), (256, 8), (256, 9)])
def test_rows_of_a_batch(cuda_dev, n, batch):
    g = gen(n)
    x = np.linspace(-1.5 * n, 1.5 * n, n)
    src = cplx(g, batch, 2, n, n)
    masks = lambda p: [MaskSpec(N.XL_MASK_LCD, p[0], p[1])]
    p = uni(g, 2, n, n)
    z = torch.linspace(20.0 * n, 30.0 * n, batch, dtype=torch.float64, device=cuda_dev)
    kw = dict(ez_mode=N.XL_EZ_VRS, nin=2)
    out = ops.rs_propagate_batched(src, x, x, 0.65, z, masks=masks(p), **kw)
    for b in (0, batch // 2, batch - 1):
        near(out[b], ops.rs_propagate(src[b], x, x, 0.0, 0.65, masks=masks(p), z_dev=z[b:b + 1], **kw), 2e-6)
