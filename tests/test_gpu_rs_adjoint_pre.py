"""Adjoint RS / VRS propagation with the pre-op adjoint in its last pass
(xl_rs_adjoint_pre) against the two separate calls (adjoint propagation, then
pre_backward), which the other tests hold to the float64 oracle: every padded
length, sides that do not divide into a block's rows or a tile's four, each
mask form, the forms that keep the separate calls, and the distance term.

Tolerances: both sides transform the same numbers with the same passes; the
pre-op's products and direction cosines round a few times in float32 (2^-24
each), so the fields agree to 1e-6 in relative L2, and the distance term, a
float64 sum of float32 products, to 2^-21 of the sum of its terms' magnitudes.
"""
import numpy as np
import pytest
import torch

from xlumina_amd import _native as N
from xlumina_amd import ops
from xlumina_amd.ops import MaskSpec

pytestmark = pytest.mark.gpu

WL, Z = 0.65, 2.1e4


def cplx(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.complex64)


def uni(g, *shape, dtype=torch.float32):
    return torch.rand(shape, generator=g, device="cuda", dtype=dtype)


def make(form, g, n):
    """(masks, ez_mode, nin, planes of the source, wanted parameter gradients)."""
    none = (False, False)
    if form == "slm":
        return [MaskSpec(N.XL_MASK_SLM, 6 * uni(g, n, n))], N.XL_EZ_NONE, 1, 1, ((True, False), none)
    if form == "slm_raw64":
        return [MaskSpec(N.XL_MASK_SLM, uni(g, n, n, dtype=torch.float64), unit=1)], N.XL_EZ_NONE, 1, 1, ((True, False), none)
    if form == "ez":
        return [], N.XL_EZ_VRS, 2, 3, (none, none)
    if form == "ez_two_planes":
        return [], N.XL_EZ_VRS, 2, 2, (none, none)
    if form == "sslm":   # (separate calls, as the rest)
        return [MaskSpec(N.XL_MASK_SSLM, 6 * uni(g, n, n), 6 * uni(g, n, n))], N.XL_EZ_VRS, 2, 3, ((True, True), none)
    if form == "sslm_raw64":
        p = [uni(g, n, n, dtype=torch.float64) for _ in range(2)]
        return [MaskSpec(N.XL_MASK_SSLM, *p, unit=3)], N.XL_EZ_VRS, 2, 3, ((False, True), none)
    if form == "lcd":
        return [MaskSpec(N.XL_MASK_LCD, uni(g, n, n), uni(g, n, n))], N.XL_EZ_VRS, 2, 3, ((True, True), none)
    if form == "slm_one_value":   # (separate calls: a sum over the pixels)
        return [MaskSpec(N.XL_MASK_SLM, uni(g, 1, dtype=torch.float64))], N.XL_EZ_NONE, 1, 1, ((True, False), none)
    raise ValueError(form)


def close(a, b, tol=1e-6):
    assert a.shape == b.shape and a.dtype == b.dtype
    a, b = a.to(torch.complex128), b.to(torch.complex128)
    assert float((a - b).norm()) <= tol * float(b.norm()), float((a - b).norm() / b.norm())


def both(form, n, need_src=True):
    g = torch.Generator(device="cuda").manual_seed(n)
    half = 1.2 * n
    x = np.linspace(-half, half, n)
    y = np.linspace(-0.9 * half, 1.1 * half, n)
    masks, ez, nin, planes, want = make(form, g, n)
    src = cplx(g, planes, n, n)
    gout = cplx(g, 3 if ez else nin, n, n)
    out = torch.full((planes, n, n), float("nan"), dtype=torch.complex64, device="cuda") if planes > nin else None
    kw = dict(masks=masks, ez_mode=ez, nin=nin, need_src=need_src, need_params=want)
    dz = dz2 = None
    if ez:
        dz, dz2 = (torch.full((ops.pre_scalar_grad_elems(n, n),), float("nan"), dtype=torch.float64, device="cuda")
                   for _ in range(2))
    base = torch.tensor([0.25], dtype=torch.float64, device="cuda") if ez else None
    got = ops.rs_propagate(gout, x, y, Z, WL, adjoint=True,
                           pre=dict(src=src, out=out, ez_dz=dz, ez_dz_base=base, **kw))
    hh = torch.empty(ops.rs_hhat_bytes(n), dtype=torch.uint8, device="cuda")   # (a call that keeps its spectrum: 2^k)
    g_pre = ops.rs_propagate(gout, x, y, Z, WL, adjoint=True, hhat=hh, hhat_mode=1)
    ref = ops.pre_backward(src, g_pre, x, y, Z, out=None if out is None else torch.empty_like(out), ez_dz=dz2,
                           ez_dz_base=base, **kw)
    if need_src:
        close(got[0], ref[0])
    else:
        assert got[0] is None
    for i in range(2):
        for j in range(2):
            assert (got[1][i][j] is None) == (ref[1][i][j] is None)
            if got[1][i][j] is not None:
                close(got[1][i][j], ref[1][i][j])
    if ez:
        e = ops.pre_forward(src, x, y, masks=masks, nin=nin).to(torch.complex128)
        X, Y = torch.from_numpy(x).cuda()[None, :], torch.from_numpy(y).cuda()[:, None]
        w = Z / torch.sqrt(X * X + Y * Y + Z * Z) ** 3
        terms = g_pre[2].abs().double() * (e[0].abs() * X.abs() + e[1].abs() * Y.abs()) * w
        assert abs(float(dz[0]) - float(dz2[0])) <= 2.0 ** -21 * float(terms.sum()) + 1e-15


FORMS = ["slm", "slm_raw64", "ez", "ez_two_planes"]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("n", [2, 31, 33, 64, 65, 127, 129, 250, 257, 511, 514, 1023])
def test_fused_matches_separate_calls(form, n):
    both(form, n)


@pytest.mark.parametrize("form", ["slm", "ez"])
@pytest.mark.parametrize("n", [1025, 2048])
def test_longest_transforms(form, n):
    both(form, n)


@pytest.mark.parametrize("form", ["slm", "sslm"])
def test_parameter_gradients_alone(form):
    both(form, 130, need_src=False)


@pytest.mark.parametrize("form", ["sslm", "sslm_raw64", "lcd", "slm_one_value"])
def test_forms_of_the_separate_calls(form):
    both(form, 130)


def test_refused():
    x = np.linspace(-50.0, 50.0, 32)
    f = torch.zeros((1, 32, 32), dtype=torch.complex64, device="cuda")
    pre = dict(src=f, masks=[], ez_mode=N.XL_EZ_NONE, nin=1, need_src=True, need_params=((False,) * 2,) * 2, out=None,
               ez_dz=None, ez_dz_base=None)
    with pytest.raises(ValueError):
        ops.rs_propagate(f, x, x, Z, WL, pre=pre)   # a forward call
    with pytest.raises(ValueError):
        ops.rs_propagate(f, x, x, Z, WL, adjoint=True, pre=dict(pre, src=torch.zeros((1, 16, 16), dtype=torch.complex64,
                                                                                   device="cuda")))
