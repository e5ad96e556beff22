"""The streaming kernels that load several pixels per thread (splitter, its
backward, the 4f loss) at plane sizes around their groups and launch limits,
against float64.

Tolerances: a splitter output is four products of float32 values and rounded
coefficients (1e-6 in relative L2); the angle gradient and the losses are
float32 sums, wrong by at most (terms per thread + 16) 2^-24 of the sum of the
terms' magnitudes, below 1e-5 of it at these sizes.  The loss's difference
|E|^2 - T may cancel, so its errors are measured against |E|^2 + T.
"""
import numpy as np
import pytest
import torch

from xlumina_amd import ops
from xlumina_amd import optical_elements as OE

pytestmark = pytest.mark.gpu

# one pixel; around a block, a group of blocks and 512 blocks of one pixel a thread; several groups per thread
SHAPES = [(1, 1), (1, 255), (3, 171), (32, 32), (33, 31), (362, 362), (363, 361), (725, 723), (1500, 1499)]


def rel(a, b):
    return float((a.to(torch.complex128) - b).norm() / b.norm())


@pytest.mark.parametrize("shape", SHAPES)
def test_splitter_and_its_backward(shape):
    g = torch.Generator(device="cuda").manual_seed(shape[0] * 4096 + shape[1])
    f = torch.randn((4, 3, *shape), generator=g, device="cuda", dtype=torch.complex64)
    a, b = (f[i].clone().requires_grad_(True) for i in range(2))
    th = torch.tensor([0.41], dtype=torch.float64, device="cuda", requires_grad=True)
    c, d = OE._SplitterTheta.apply(a, b, th, 1)
    got = torch.autograd.grad((c, d), (a, b, th), (f[2], f[3]))
    A, B, G, H = (f[i, :2].to(torch.complex128) for i in range(4))
    co, si = np.cos(0.41), np.sin(0.41)
    R, T, dR, dT = si - 0.01 * co, 0.99 * co, co + 0.01 * si, -0.99 * si
    assert rel(c[:2].detach(), R * A + 1j * T * B) <= 1e-6 and rel(d[:2].detach(), 1j * T * A + R * B) <= 1e-6
    assert rel(got[0][:2], R * G - 1j * T * H) <= 1e-6 and rel(got[1][:2], -1j * T * G + R * H) <= 1e-6
    for t in (c, d, got[0], got[1]):
        assert float(t[2].detach().abs().max()) == 0.0
    terms = torch.stack([G.conj() * (dR * A + 1j * dT * B), H.conj() * (1j * dT * A + dR * B)])
    mags = (G.abs() + H.abs()) * (A.abs() + B.abs())
    assert abs(float(got[2]) - float(terms.real.sum())) <= 1e-5 * float(mags.sum())


@pytest.mark.parametrize("shape", SHAPES)
def test_mse_intensity(shape):
    g = torch.Generator(device="cuda").manual_seed(shape[0] * 4096 + shape[1])
    e = torch.randn((2, *shape), generator=g, device="cuda", dtype=torch.complex64)
    tgt = torch.rand(shape, generator=g, device="cuda")
    grad, loss = torch.empty_like(e), torch.empty(2, device="cuda")
    ops.mse_intensity(e, tgt, grad=grad, loss=loss)
    E = e.to(torch.complex128)
    d = E.abs() ** 2 - tgt.double()
    n = shape[0] * shape[1]
    big = E.abs() ** 2 + tgt.double()
    assert float((grad.to(torch.complex128) - 4 * d * E / n).norm()) <= 1e-6 * float((4 * big * E / n).norm())
    assert float(((loss.double() - (d * d).sum((1, 2)) / n).abs() * n / (big * big).sum((1, 2))).max()) <= 1e-5
