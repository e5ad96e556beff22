"""Row / column blocks of the RS kernels at the sizes where they can go wrong:
both sides of every padded length, sides that do not divide into a block's
rows or a tile's four, against the float64 oracle (relative L2 <= 1e-5, the
FP32 paths' bar), with the batched launch and the distance gradient's column
sums at the same sizes.
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
TOL = 1e-5

SIZES = [2, 5, 31, 33, 63, 66, 127, 130, 255, 258, 511, 513, 514, 640, 641, 768, 769, 1023, 1026, 1280, 1281, 1536]


@pytest.mark.parametrize("n", SIZES)
def test_block_edges_vs_oracle(cuda_dev, n):
    rng = np.random.default_rng(n)
    x, y = R.space(3.0 * n, n)
    ex, ey = rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))
    a, b = rng.uniform(-np.pi, np.pi, (2, n, n)).astype(np.float32)
    dev = lambda v, t: torch.tensor(np.ascontiguousarray(v), dtype=t, device=cuda_dev)
    z, wl = 40.0 * n, 0.65
    masks = [MaskSpec(N.XL_MASK_SSLM, dev(a, torch.float32), dev(b, torch.float32))]
    src = dev(np.stack([ex, ey]), torch.complex64)
    out, inten = ops.rs_propagate(src, x, y, z, wl, masks=masks, ez_mode=N.XL_EZ_VRS, nin=2, intensity=True)
    mx, my = ex * np.exp(1j * a.astype(np.float64)), ey * np.exp(1j * b.astype(np.float64))
    ref = np.stack(R.vrs_propagation(mx, my, x, y, wl, z)[0])
    assert rel_l2(out.cpu().numpy(), ref) < TOL
    assert rel_l2(inten.cpu().numpy(), np.sum(np.abs(ref) ** 2, axis=0)) < TOL
    # one component, and the adjoint identity <g, A f> = <A^H g, f>
    f, g = src[:1], src[1:]
    af = ops.rs_propagate(f, x, y, z, wl)
    assert rel_l2(af[0].cpu().numpy(), R.rs_propagation(ex, x, y, wl, z)[0]) < TOL
    hg = ops.rs_propagate(g, x, y, z, wl, adjoint=True)
    lhs = torch.sum(g.to(torch.complex128).conj() * af.to(torch.complex128))
    rhs = torch.sum(hg.to(torch.complex128).conj() * f.to(torch.complex128))
    scale = float(torch.linalg.vector_norm(g) * torch.linalg.vector_norm(af))
    assert abs(complex(lhs - rhs)) <= 1e-5 * scale


@pytest.mark.parametrize("n", [513, 700, 1100, 1300])
def test_plain_and_kept_spectra_agree(cuda_dev, n):
    """A plain call runs at the shortest length, one that keeps its kernel
    spectrum at the power of two: the same propagation to rounding (each within
    1e-6 of float64, so 2e-6 apart at most), with float64 and one-value mask
    parameters and masks in both stages."""
    rng = np.random.default_rng(n)
    x, y = R.space(1.17 * n, n)
    f = rng.standard_normal((3, n, n)) + 1j * rng.standard_normal((3, n, n))
    src = torch.tensor(f.astype(np.complex64), device=cuda_dev)
    p = torch.tensor(rng.uniform(0, 1, (2, n, n)), dtype=torch.float64, device=cuda_dev)
    v = torch.tensor([0.3], dtype=torch.float64, device=cuda_dev)
    masks = [MaskSpec(N.XL_MASK_SSLM, p[0], p[1], unit=3), MaskSpec(N.XL_MASK_LCD, v, v)]
    hh = torch.empty(ops.rs_hhat_bytes(n), dtype=torch.uint8, device=cuda_dev)
    for kw in (dict(masks=masks, ez_mode=N.XL_EZ_VRS, nin=2), dict(masks=masks, nin=3), dict(nin=3, adjoint=True, masks=())):
        a = ops.rs_propagate(src, x, y, 4e4, 0.65, **kw)
        b = ops.rs_propagate(src, x, y, 4e4, 0.65, hhat=hh, hhat_mode=1, **kw)
        assert rel_l2(a.cpu().numpy(), b.cpu().numpy()) < 2e-6


@pytest.mark.parametrize("n", [31, 130, 514])
def test_block_edges_batched_equals_alone(cuda_dev, n):
    """Members of a batch run in blocks of their own: the same bits as alone."""
    g = torch.Generator(device="cuda").manual_seed(n)
    x, y = R.space(3.0 * n, n)
    src = torch.complex(torch.randn((3, 2, n, n), generator=g, device=cuda_dev),
                        torch.randn((3, 2, n, n), generator=g, device=cuda_dev))
    z = torch.tensor([30.0 * n, 41.0 * n, 52.0 * n], dtype=torch.float64, device=cuda_dev)
    out, inten = ops.rs_propagate_batched(src, x, y, 0.65, z, ez_mode=N.XL_EZ_VRS, nin=2, intensity=True)
    for b in range(3):
        o, i = ops.rs_propagate(src[b], x, y, 0.0, 0.65, ez_mode=N.XL_EZ_VRS, nin=2, intensity=True, z_dev=z[b:b + 1])
        assert torch.equal(out[b], o) and torch.equal(inten[b], i)


@pytest.mark.parametrize("n,comps", [(31, 1), (66, 3), (130, 3), (514, 1), (1026, 1)])
def test_block_edges_distance_gradient(cuda_dev, n, comps):
    """The column pass's distance-gradient sums (prebuilt and own derivative
    spectra) against the derivative propagation dotted with the cotangent,
    <= 2e-5 of |d||g|."""
    gen = torch.Generator(device="cuda").manual_seed(n)
    x, y = R.space(3.0 * n, n)
    c64 = lambda: torch.complex(torch.randn((comps, n, n), generator=gen, device=cuda_dev),
                                torch.randn((comps, n, n), generator=gen, device=cuda_dev))
    src, g = c64(), c64()
    z, wl = 40.0 * n, 0.65
    hh = torch.empty(ops.rs_hhat_bytes(n), dtype=torch.uint8, device=cuda_dev)
    sp = torch.empty(ops.rs_spec_bytes(n, comps), dtype=torch.uint8, device=cuda_dev)
    ops.rs_propagate(src, x, y, z, wl, hhat=hh, hhat_mode=1, spec=sp, spec_mode=1, spec_grads=3)
    refs = []
    for kind in (1, 2):
        d = ops.rs_propagate(src, x, y, z, wl, kernel_dz=kind)
        dot = float(torch.sum(torch.real(g.to(torch.complex128).conj() * d.to(torch.complex128))))
        refs.append((dot, float(torch.linalg.vector_norm(d) * torch.linalg.vector_norm(g))))
    for bits in (3, 3 | N.XL_RS_SPEC_PREBUILT, 1 | N.XL_RS_SPEC_PREBUILT, 2):
        out = torch.zeros(2, dtype=torch.float64, device=cuda_dev)
        ops.rs_propagate(g, x, y, z, wl, adjoint=True, hhat=hh, hhat_mode=2, spec=sp, spec_mode=2, spec_grads=bits,
                         grad_out=out)
        for i in range(2):
            if bits >> i & 1:
                assert abs(float(out[i]) - refs[i][0]) <= 2e-5 * refs[i][1], (bits, i)
