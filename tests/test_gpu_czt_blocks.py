"""Row / column passes of the Bluestein CZT at the sizes where they can go
wrong (both sides of each FFT length and of its zero-half forms, sides that do
not divide into a tile or a column pair, one and several components, batches),
against the float64 oracle (relative L2 <= 1e-5, the FP32 paths' bar); and the
rule that picks a transform's form.
"""
import numpy as np
import pytest
import torch

from oracle import xlumina_ref as R
from tests.conftest import rel_l2
from xlumina_amd import _native as N
from xlumina_amd import ops
from xlumina_amd.ops import MaskSpec

TOL = 1e-5
# (n, my, mx): zero-half lengths 64..4096, full lengths (n or m above half), 3 * 2^k columns, odd sides
SIZES = [(17, 9, 8), (32, 31, 30), (33, 20, 31), (65, 40, 63), (100, 28, 30), (129, 130, 127), (250, 101, 99),
         (257, 250, 64), (400, 61, 33), (513, 500, 258), (700, 20, 130), (777, 301, 301), (1000, 24, 510), (1025, 66, 90),
         (1030, 1021, 34), (2047, 50, 34)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,my,mx", SIZES)
def test_czt_edges_vs_oracle(cuda_dev, n, my, mx):
    rng = np.random.default_rng(n + my)
    x, y = R.space(2.0 * n, n)
    xo, yo = np.linspace(-0.3 * n, 0.35 * n, mx), np.linspace(-0.4 * n, 0.3 * n, my)
    ex, ey = rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))
    src = torch.tensor(np.stack([ex, ey]).astype(np.complex64), device=cuda_dev)
    z, wl = 3e4, 0.635
    g = ops.czt_geometry(x, y, xo, yo, z, wl)
    one = ops.czt(src[:1], g, form="bluestein")
    assert rel_l2(one[0].cpu().numpy(), R.czt(ex, x, y, wl, z, xo, yo)) < TOL
    three = ops.czt(src, g, ez_mode=N.XL_EZ_VCZT, nin=2, form="bluestein")
    assert rel_l2(three.cpu().numpy(), np.stack(R.vczt(ex, ey, x, y, wl, z, xo, yo))) < TOL
    # the adjoint identity <g, A f> = <A^H g, f>, one and three components
    gen = torch.Generator(device="cuda").manual_seed(n)
    for c, f in ((1, src[:1]), (2, src)):
        cot = torch.complex(torch.randn((c, my, mx), generator=gen, device=cuda_dev),
                            torch.randn((c, my, mx), generator=gen, device=cuda_dev))
        af = ops.czt(f, g, form="bluestein")
        hg = ops.czt(cot, g, adjoint=True, form="bluestein")
        lhs = torch.sum(cot.to(torch.complex128).conj() * af.to(torch.complex128))
        rhs = torch.sum(hg.to(torch.complex128).conj() * f.to(torch.complex128))
        assert abs(complex(lhs - rhs)) <= 1e-5 * float(torch.linalg.vector_norm(cot) * torch.linalg.vector_norm(af))


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,batch", [(33, 20, 2), (250, 99, 5), (1025, 66, 4)])
def test_czt_batched_equals_alone(cuda_dev, n, m, batch):
    """Members of a batch run in blocks of their own; from 4 members on the
    plane factors come from tables, so the bar is rounding (1e-6)."""
    gen = torch.Generator(device="cuda").manual_seed(n)
    x, y = R.space(2.0 * n, n)
    xo = np.linspace(-0.3 * n, 0.35 * n, m)
    g = ops.czt_geometry(x, y, xo, xo, 3e4, 0.635)
    src = torch.complex(torch.randn((batch, 1, n, n), generator=gen, device=cuda_dev),
                        torch.randn((batch, 1, n, n), generator=gen, device=cuda_dev))
    ph = torch.rand((batch, n, n), generator=gen, device=cuda_dev)
    out = ops.czt(src, g, masks=[MaskSpec(N.XL_MASK_SLM, ph)], batch=batch)
    for b in range(batch):
        alone = ops.czt(src[b], g, masks=[MaskSpec(N.XL_MASK_SLM, ph[b])], form="bluestein")
        assert rel_l2(out[b].cpu().numpy(), alone.cpu().numpy()) < 1e-6


def _geometry(n, m, hna=False):
    x, y = R.space(1800.0, n)
    xo = np.linspace(-10.0, 10.0, m)
    return ops.hna_geometry(x, y, xo, xo, 0.635, 1800.0, 2000.0) if hna else ops.czt_geometry(x, y, xo, xo, 3e4, 0.635)


@pytest.mark.parametrize("n,m,ncomp,form", [(2048, 128, 3, "gemm"), (2048, 129, 3, "bluestein"), (1537, 64, 3, "gemm"),
                                            (1536, 64, 3, "bluestein"), (2048, 64, 1, "bluestein"),
                                            (256, 64, 3, "bluestein")])
def test_auto_form_by_size(n, m, ncomp, form):
    assert ops.resolve_czt_form(_geometry(n, m), None, ncomp) == form
    assert ops.resolve_czt_form(_geometry(n, m), "gemm", ncomp) == "gemm"
    assert ops.resolve_czt_form(_geometry(n, m), "bluestein", ncomp) == "bluestein"


@pytest.mark.parametrize("n,m,form", [(256, 160, "gemm"), (2048, 160, "gemm"), (256, 161, "bluestein")])
def test_auto_form_of_the_lens(n, m, form):
    assert ops.resolve_czt_form(_geometry(n, m, hna=True)) == form


@pytest.mark.gpu
@pytest.mark.parametrize("n,m", [(1536, 64), (1538, 128)])
def test_auto_form_vs_oracle(cuda_dev, n, m):
    """Both sides of the rule's line: <= 1e-5 in the FP32 form, <= 1e-4 in the
    split-BF16 form (each form's bar)."""
    rng = np.random.default_rng(n)
    x, y = R.space(1.17 * n, n)
    xo = np.linspace(-100.0, 100.0, m)
    ex, ey = rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))
    src = torch.tensor(np.stack([ex, ey]).astype(np.complex64), device=cuda_dev)
    g = ops.czt_geometry(x, y, xo, xo, 3e4, 0.635)
    out = ops.czt(src, g, ez_mode=N.XL_EZ_VCZT, nin=2)
    bar = 1e-5 if ops.resolve_czt_form(g) == "bluestein" else 1e-4
    assert rel_l2(out.cpu().numpy(), np.stack(R.vczt(ex, ey, x, y, 0.635, 3e4, xo, xo))) < bar
