"""State that differentiated propagations share: kernel spectra by grid and
distance, CZT tables by geometry.  What may be shared, and what may not.
"""
import ctypes
import threading

import numpy as np
import pytest
import torch

from oracle import xlumina_ref as R
from tests.conftest import rel_l2
from xlumina_amd import _native as N
from xlumina_amd import autograd as AG
from xlumina_amd import ops

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


def test_spectra_key_follows_the_launch_scope(monkeypatch):
    x = torch.linspace(-8.0, 8.0, 16, dtype=torch.float64)
    keys = []
    for scope in ((0, 0), (1, 0), (1, 7), (1, 8), (2, 0)):   # (stream, graph capture)
        monkeypatch.setattr(ops, "launch_scope", lambda dev: scope, raising=False)
        keys.append(AG._spectra_key(_rs_config(x), None, 16, 1, CPU)[0])
    assert len(set(keys)) == len(keys)


def test_capture_id_of_the_default_stream():
    assert ops.launch_scope(CPU) == (0, 0)
    cid = ctypes.c_uint64(5)
    N.check(N.load().xl_capture_id(None, ctypes.byref(cid)))
    assert cid.value == 0
    with pytest.raises(ValueError):
        N.check(N.load().xl_capture_id(None, None))


def _c64(gen, *shape):
    return torch.view_as_complex(torch.randn((*shape, 2), generator=gen, device=gen.device))


@pytest.mark.gpu
def test_propagations_on_two_streams_build_their_own_spectra(cuda_dev):
    """Forward and adjoint on two streams at once: the bits of the same calls
    one after the other."""
    n = 160
    x = np.linspace(-150.0, 150.0, n)
    gen = torch.Generator(device=cuda_dev).manual_seed(5)
    src, w = _c64(gen, 2, 1, n, n), torch.rand((2, n, n), generator=gen, device=cuda_dev)

    def step(i):
        s = src[i].clone().requires_grad_(True)
        out = AG.rs(s, x, x, 700.0, 0.65)
        return out, torch.autograd.grad((w[i] * out.abs() ** 2).sum(), s, retain_graph=True)[0]

    AG._SHARED_SPECTRA.clear()
    one = [step(i) for i in range(2)]
    assert len(AG._SHARED_SPECTRA) == 1
    torch.cuda.synchronize()
    AG._SHARED_SPECTRA.clear()
    streams = [torch.cuda.Stream(cuda_dev) for _ in range(2)]
    two = []
    for i, st in enumerate(streams):
        with torch.cuda.stream(st):
            two.append(step(i))
    assert len(AG._SHARED_SPECTRA) == 2
    torch.cuda.synchronize()
    for (a, ga), (b, gb) in zip(one, two):
        assert torch.equal(a.detach(), b.detach()) and torch.equal(ga, gb)


@pytest.mark.gpu
def test_captured_propagation_builds_its_own_spectra(cuda_dev):
    """A step captured while an eager step's output over the same distance is
    alive on the capture's stream, replayed after that output and its memory
    are gone: the eager values, each time."""
    n = 96
    x = np.linspace(-150.0, 150.0, n)
    gen = torch.Generator(device=cuda_dev).manual_seed(6)
    src = _c64(gen, 1, n, n).requires_grad_(True)
    st = torch.cuda.Stream(cuda_dev)
    st.wait_stream(torch.cuda.current_stream(cuda_dev))
    with torch.cuda.stream(st):
        eager = AG.rs(src, x, x, 700.0, 0.65)
        ref = eager.detach().clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        out = AG.rs(src, x, x, 700.0, 0.65)
    del eager
    for _ in range(3):
        junk = torch.full((64 << 20,), float("nan"), device=cuda_dev)   # takes what the eager step held
        with torch.cuda.stream(st):
            side = torch.full((4 << 20,), float("nan"), device=cuda_dev)
            out.detach().zero_()
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.detach(), ref)
        del junk, side


def _czt_config(n=16):
    x = np.linspace(-100.0, 100.0, n)
    xo = np.linspace(-9.0, 9.0, 10)
    return AG.CZTConfig(ops.czt_geometry(x, x, xo, xo, 3e4, 0.65), N.XL_EZ_NONE, 1, N.XL_CZT_RS)


def test_staged_tables_follow_the_launch_scope_and_thread(monkeypatch):
    shares = [AG._staged_tables(_czt_config(), CPU)]
    assert AG._staged_tables(_czt_config(), CPU) is shares[0]
    for scope in ((1, 0), (1, 7), (2, 0)):
        monkeypatch.setattr(ops, "launch_scope", lambda dev: scope)
        shares.append(AG._staged_tables(_czt_config(), CPU))
    worker = threading.Thread(target=lambda: shares.append(AG._staged_tables(_czt_config(), CPU)))
    worker.start()
    worker.join()
    assert len({id(s) for s in shares}) == 5


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["streams", "threads"])
def test_zooms_of_one_geometry_at_once(cuda_dev, how):
    """Differentiated zooms of one geometry on two streams, and from two
    threads on one stream: the bits of the same calls one after the other."""
    n, m = 300, 200
    x = np.linspace(-900.0, 900.0, n)
    xo = np.linspace(-90.0, 90.0, m)
    gen = torch.Generator(device=cuda_dev).manual_seed(8)
    src, w = _c64(gen, 2, 2, n, n), torch.rand((2, m, m), generator=gen, device=cuda_dev)

    def forward(i):
        s = src[i].clone().requires_grad_(True)
        geom = ops.czt_geometry(x, x, xo, xo, 3e4, 0.65)
        return s, [AG.czt(s, geom, nin=2, form="bluestein") for _ in range(4)]

    def step(i):
        s, outs = forward(i)
        return [o.detach() for o in outs], torch.autograd.grad(sum((w[i] * o.abs() ** 2).sum() for o in outs), s)[0]

    ref = [step(i) for i in range(2)]
    torch.cuda.synchronize()
    got = [None, None]

    def on(i, st):
        with torch.cuda.stream(st):
            got[i] = step(i)

    if how == "streams":
        streams = [torch.cuda.Stream(cuda_dev) for _ in range(2)]
        for i in range(2):
            on(i, streams[i])
    else:
        st = torch.cuda.Stream(cuda_dev)
        workers = [threading.Thread(target=on, args=(i, st)) for i in range(2)]
        for t in workers:
            t.start()
        for t in workers:
            t.join()
    torch.cuda.synchronize()
    for (outs, g), (outs2, g2) in zip(ref, got):
        assert all(torch.equal(a, b) for a, b in zip(outs, outs2)) and torch.equal(g, g2)


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
