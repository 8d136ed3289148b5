"""Scratch kept between calls: pooled plans of the autograd P2M, pinned status
words."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mods():
    from ppm_legacy_amd import autograd, core
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return autograd, core


def _inputs(core, n, N, seed, dim=3):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.rand((n, dim), dtype=torch.float64, device="cuda", generator=g).requires_grad_(True)
    u = torch.randn((n, 2), dtype=torch.float64, device="cuda", generator=g).requires_grad_(True)
    mesh = core.Mesh(dim, N + 1)
    return x, u, mesh, torch.randn(mesh.compact_shape(2), dtype=torch.float64, device="cuda", generator=g)


def _grads(autograd, case):
    x, u, mesh, g = case
    f = autograd.p2m(x, u, mesh)
    return (f.detach(),) + torch.autograd.grad(f, (x, u), g)


def test_graph_plans_pooled(mods):
    """Graphs of different sizes one after another, two alive at once, on two
    streams and freed in either order: every result as from a new plan."""
    autograd, core = mods
    cases = [_inputs(core, n, N, s, d) for n, N, s, d in ((5000, 16, 1, 3), (300, 8, 2, 3), (20000, 90, 3, 2))]
    want = []
    for c in cases:
        autograd.release_plans()
        want.append(_grads(autograd, c))
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for rep in range(4):
        for c, w in zip(cases, want):
            with torch.cuda.stream(side if rep % 2 else torch.cuda.current_stream()):
                got = _grads(autograd, c)
            torch.cuda.current_stream().wait_stream(side)
            assert all(torch.equal(a, b) for a, b in zip(got, w))
        torch.cuda.synchronize()
    assert 0 < len(autograd._pool[0]) <= 3
    f = [autograd.p2m(c[0], c[1], c[2]) for c in cases]           # three graphs alive
    for i in (1, 2, 0):
        gx, gu = torch.autograd.grad(f[i], cases[i][:2], cases[i][3])
        assert torch.equal(gx, want[i][1]) and torch.equal(gu, want[i][2])
        f[i] = None
    autograd.release_plans()
    assert not autograd._pool


def test_graph_plans_bounded(mods, monkeypatch):
    """Scratch over the pool's bound is freed with its graph."""
    autograd, core = mods
    autograd.release_plans()
    monkeypatch.setattr(autograd, "POOL_BYTES", 1 << 10)
    _grads(autograd, _inputs(core, 1000, 12, 5))
    assert not autograd._pool.get(0)


def test_graph_plans_from_threads(mods):
    """Threads with a stream each share the pool."""
    autograd, core = mods
    cases = [_inputs(core, 4000 + i, 20, 10 + i) for i in range(4)]
    want = [_grads(autograd, c) for c in cases]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(10):
                got = _grads(autograd, cases[i])
                s.synchronize()
                if not all(torch.equal(a, b) for a, b in zip(got, want[i])):
                    bad.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    autograd.release_plans()


def test_noncontiguous_positions(mods):
    """Positions that the forward copied: the gradients use them from the graph."""
    autograd, core = mods
    x, u, mesh, g = _inputs(core, 3000, 40, 7, 2)
    want = _grads(autograd, (x, u, mesh, g))
    xt = x.detach().t().contiguous().t().requires_grad_(True)
    assert not xt.is_contiguous()
    f = autograd.p2m(xt, u, mesh)
    torch.empty(3000 * 2, dtype=torch.float64, device="cuda").fill_(9.0)
    gx, gu = torch.autograd.grad(f, (xt, u), g)
    assert torch.equal(gx, want[1]) and torch.equal(gu, want[2])


def test_many_plans(mods):
    """More plans than pinned slots: the rest copy their status words."""
    _, core = mods
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand((100, 3), dtype=torch.float64, device="cuda", generator=g)
    u = torch.ones((100, 1), dtype=torch.float64, device="cuda")
    mesh = core.Mesh(3, 9)
    plans, ref = [], None
    for i in range(260):
        f = torch.empty(mesh.compact_shape(1), dtype=torch.float64, device="cuda")
        plans.append(core.p2m(mesh, x, u, f, [0] * 3))
        ref = f if ref is None else ref
        assert torch.equal(f, ref)
