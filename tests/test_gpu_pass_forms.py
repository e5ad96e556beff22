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


@pytest.mark.parametrize("n", [1537, 2047])
def test_longest_length(cuda_dev, n):
    """The first side past the shorter lengths and the last odd one."""
    g = gen(n)
    x = np.linspace(-1.2 * n, 1.2 * n, n)
    f, c = cplx(g, 1, n, n), cplx(g, 1, n, n)
    af = ops.rs_propagate(f, x, x, 4e4, 0.65)
    adjoint_identity(f, af, c, ops.rs_propagate(c, x, x, 4e4, 0.65, adjoint=True))
    three = ops.rs_propagate(f.expand(3, n, n).contiguous(), x, x, 4e4, 0.65)
    for i in range(3):
        near(three[i:i + 1], af, 2e-6)


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


# columns staged through LDS or not: outputs within, at and above the inputs (full and zero-half lengths 128..1024)
@pytest.mark.parametrize("n,m", [(50, 30), (64, 66), (100, 28), (120, 130), (130, 120), (61, 400), (200, 300), (300, 200),
                                 (99, 250), (100, 200), (100, 199), (100, 500), (300, 700), (512, 512)])
def test_column_forms(cuda_dev, n, m):
    rng = np.random.default_rng(n + m)
    x, y = R.space(2.0 * n, n)
    xo = np.linspace(-0.3 * n, 0.35 * n, m)
    e = rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))
    src = torch.tensor(e.astype(np.complex64), device=cuda_dev)
    geom = ops.czt_geometry(x, y, xo, xo, 3e4, 0.635)
    out = ops.czt(src, geom, ez_mode=N.XL_EZ_VCZT, nin=2, form="bluestein")
    assert rel_l2(out.cpu().numpy(), np.stack(R.vczt(e[0], e[1], x, y, 0.635, 3e4, xo, xo))) < 1e-5
    cot = cplx(gen(n), 2, m, m)
    adjoint_identity(src, ops.czt(src, geom, form="bluestein"), cot, ops.czt(cot, geom, adjoint=True, form="bluestein"))


# 64 MB of tiles: columns of the batch staged, a member's alone direct; then rows of one component whose plane factors
# come from a table, most of the row being input or not
@pytest.mark.parametrize("n,m,batch", [(1024, 1024, 8), (1023, 1009, 9), (700, 300, 4), (640, 300, 4), (641, 300, 4),
                                       (1500, 500, 4)])
def test_forms_of_a_batch(cuda_dev, n, m, batch):
    g = gen(n)
    x, xo = np.linspace(-900.0, 900.0, n), np.linspace(-400.0, 390.0, m)
    geom = ops.czt_geometry(x, x, xo, xo, 3e4, 0.635)
    src, cot, ph = cplx(g, batch, 1, n, n), cplx(g, batch, 1, m, m), uni(g, batch, n, n)
    out = ops.czt(src, geom, masks=[MaskSpec(N.XL_MASK_SLM, ph)], batch=batch)
    adj = ops.czt(cot, geom, adjoint=True, batch=batch)
    for b in (0, batch - 1):
        near(out[b], ops.czt(src[b], geom, masks=[MaskSpec(N.XL_MASK_SLM, ph[b])], form="bluestein"), 2e-6)
        near(adj[b], ops.czt(cot[b], geom, adjoint=True, form="bluestein"), 2e-6)


# up to 256 rows of 4096 points: three components side by side; more: one after the other
@pytest.mark.parametrize("m", [2, 3, 255, 256, 257])
@pytest.mark.parametrize("hna", [False, True])
def test_few_long_rows(cuda_dev, m, hna):
    n = 2048
    x = np.linspace(-1800.0, 1800.0, n)
    xo, yo = np.linspace(-9.0, 8.0, 200), np.linspace(-8.0, 9.0, m)
    geom = (ops.hna_geometry(x, x, xo, yo, 0.635, 1800.0, 2000.0) if hna else ops.czt_geometry(x, x, xo, yo, 3e4, 0.635))
    g = gen(m)
    cot = cplx(g, 3, m, 200)
    got = ops.czt(cot, geom, adjoint=True, form="bluestein")
    for c in range(3):   # a component alone takes the one-buffer rows
        if hna:
            only = torch.zeros_like(cot)
            only[c] = cot[c]
            one = ops.czt(only, geom, adjoint=True, form="bluestein")
            assert float(one[[i for i in range(3) if i != c]].abs().max()) == 0.0
            near(got[c], one[c], 2e-6)
        else:
            near(got[c:c + 1], ops.czt(cot[c:c + 1], geom, adjoint=True, form="bluestein"), 2e-6)
    f = cplx(g, 3, n, n)
    af = ops.czt(f, geom, form="bluestein") if not hna else None
    if af is not None:
        adjoint_identity(f, af, cot, got)


@pytest.mark.parametrize("n", [200, 256, 258])
def test_long_rows_of_a_small_pupil(cuda_dev, n):
    """Few input rows onto a wide window: 4096-point rows of three components."""
    rng = np.random.default_rng(n)
    x, y = R.space(1800.0, n)
    xo = np.linspace(-60.0, 60.0, 1900)
    e = rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))
    src = torch.tensor(e.astype(np.complex64), device=cuda_dev)
    out = ops.czt(src, ops.hna_geometry(x, y, xo, xo, 0.65, 1800.0, 2000.0), nin=2, form="bluestein")
    ref = np.stack(R.vczt_objective_lens(e[0], e[1], x, y, 0.65, 1800.0, 2000.0, xo, xo))
    assert rel_l2(out.cpu().numpy(), ref) < 1e-5
    out = ops.czt(src, ops.czt_geometry(x, y, xo, xo, 3e4, 0.65), ez_mode=N.XL_EZ_VCZT, nin=2, form="bluestein")
    assert rel_l2(out.cpu().numpy(), np.stack(R.vczt(e[0], e[1], x, y, 0.65, 3e4, xo, xo))) < 1e-5


@pytest.mark.parametrize("n", [31, 130, 514])
def test_distance_term_of_the_joined_adjoint(cuda_dev, n):
    """The joined adjoint call on a device distance, its distance term started
    from the column pass's partial sums, against the separate calls started
    from their sum: float32 products summed in float64, 2^-21 of the terms."""
    g = gen(n)
    x, y = np.linspace(-1.2 * n, 1.2 * n, n), np.linspace(-1.1 * n, 1.3 * n, n)
    z = torch.tensor([2.1e4], dtype=torch.float64, device=cuda_dev)
    src, gout = cplx(g, 2, n, n), cplx(g, 3, n, n)
    hh = torch.empty(ops.rs_hhat_bytes(n), dtype=torch.uint8, device=cuda_dev)
    sp = torch.empty(ops.rs_spec_bytes(n, 3), dtype=torch.uint8, device=cuda_dev)
    ops.rs_propagate(src, x, y, 0.0, 0.65, ez_mode=N.XL_EZ_VRS, nin=2, z_dev=z, hhat=hh, hhat_mode=1, spec=sp, spec_mode=1,
                     spec_grads=1)
    adj = dict(adjoint=True, z_dev=z, hhat=hh, hhat_mode=2, spec=sp, spec_mode=2)
    dz, dz2 = (torch.full((ops.pre_scalar_grad_elems(n, n),), float("nan"), dtype=torch.float64, device=cuda_dev)
               for _ in range(2))
    pre = dict(ez_mode=N.XL_EZ_VRS, nin=2, masks=[], need_src=True, need_params=((False,) * 2,) * 2, out=None)
    got, _ = ops.rs_propagate(gout, x, y, 0.0, 0.65, spec_grads=1 | N.XL_RS_SPEC_PREBUILT | N.XL_RS_SPEC_PARTIALS,
                              pre=dict(pre, src=src, ez_dz=dz, ez_dz_base=ops.rs_spec_partials(sp, n, 3, 0)), **adj)
    sums = torch.empty(2, dtype=torch.float64, device=cuda_dev)
    g_pre = ops.rs_propagate(gout, x, y, 0.0, 0.65, spec_grads=1 | N.XL_RS_SPEC_PREBUILT, grad_out=sums, **adj)
    ref, _ = ops.pre_backward(src, g_pre, x, y, 0.0, z_dev=z, ez_dz=dz2, ez_dz_base=sums[:1], **pre)
    near(got, ref, 1e-6)
    X, Y = torch.from_numpy(x).cuda()[None, :], torch.from_numpy(y).cuda()[:, None]
    w = float(z) / torch.sqrt(X * X + Y * Y + z * z) ** 3
    e = src.to(torch.complex128)
    terms = g_pre[2].abs().double() * (e[0].abs() * X.abs() + e[1].abs() * Y.abs()) * w
    assert abs(float(dz[0]) - float(dz2[0])) <= 2.0 ** -21 * float(terms.sum()) + 1e-12 * abs(float(sums[0]))
