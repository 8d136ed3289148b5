"""The pool of the autograd P2M's plans, with the device taken out: which plan
a graph gets, what it waits for and what goes back."""
import types

import pytest
import torch

from ppm_legacy_amd import _lib, autograd, core


class Stream:
    def __init__(self, device, handle=0):
        self.device_index, self.cuda_stream, self.waits = device, handle, []

    def wait_event(self, event):
        self.waits.append(event)


class Event:
    def __init__(self):
        self.stream = None

    def record(self, stream):
        # an event belongs to the device it is first recorded on
        assert self.stream is None or self.stream.device_index == stream.device_index
        self.stream = stream

    def synchronize(self):
        pass


class Plan:
    def __init__(self):
        self.closed = False

    def scratch_bytes(self):
        return 100

    def close(self):
        self.closed = True


class Device:
    """Stands for torch.cuda: current device and its current stream."""

    def __init__(self, monkeypatch):
        self.streams = {d: Stream(d) for d in (0, 1)}
        self.current = 0
        monkeypatch.setattr(torch.cuda, "current_device", lambda: self.current)
        monkeypatch.setattr(torch.cuda, "current_stream",
                            lambda d=None: self.streams[self.current if d is None else torch.device("cuda", d).index
                                                        if not isinstance(d, torch.device) else d.index or 0])
        monkeypatch.setattr(torch.cuda, "Event", Event)
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d=None: (1 << 40, 1 << 40), raising=False)
        monkeypatch.setattr(core, "Plan", Plan)


@pytest.fixture
def dev(monkeypatch):
    d = Device(monkeypatch)
    monkeypatch.setattr(autograd, "_pool", {})
    plans = []
    monkeypatch.setattr(core, "p2m", lambda mesh, x, u, f, lo, k, p, plan: (plans.append(plan), f.zero_()))
    monkeypatch.setattr(core, "p2m_adjoint", lambda mesh, x, u, g, lo, plan, k, p, want_u, want_x:
                        (plans.append(plan), (torch.zeros_like(u), torch.zeros_like(x)))[1])
    d.plans = plans
    return d


def _graph(mesh=core.Mesh(2, 9)):
    x = torch.rand((5, 2), dtype=torch.float64).requires_grad_(True)
    u = torch.ones((5, 1), dtype=torch.float64).requires_grad_(True)
    return autograd.p2m(x, u, mesh), (x, u)


def test_filed_under_the_device_the_work_ran_on(dev, monkeypatch):
    """The library works on the current device, wherever the tensors are: here
    on device 0 with device 1 current."""
    dev.current = 1
    ctx = types.SimpleNamespace(save_for_backward=lambda *a: None)
    up = types.SimpleNamespace(shape=(5, 1), device=torch.device("cuda", 0), contiguous=lambda: None)
    with monkeypatch.context() as m:
        empty = torch.empty
        m.setattr(torch, "empty", lambda *a, device=None, **k: empty(*a, **k))
        autograd.P2MFunction.forward(ctx, up, up, core.Mesh(2, 9), core.L.KERNEL_MP4, core.PREC_F64)
    del ctx
    assert not autograd._pool.get(0)
    (plan, event), = [e[:2] for e in autograd._pool[1]]
    assert plan is dev.plans[0] and event.stream is dev.streams[1]
    dev.current = 0
    f, _ = _graph()
    assert dev.plans[1] is not plan
    dev.current = 1
    g, _ = _graph()
    assert dev.plans[2] is plan


def test_default_streams_of_two_devices_differ(dev):
    """Both devices' default streams have the handle 0: a plan last used on
    the other device is waited for."""
    f, xu = _graph()
    dev.current = 1
    torch.autograd.grad(f.sum(), xu)     # the adjoint with device 1 current
    del f
    dev.current = 0
    (_, event), = [e[:2] for e in autograd._pool[0]]
    assert event.stream is dev.streams[1]
    g, _ = _graph()
    assert dev.plans[-1] is dev.plans[0] and dev.streams[0].waits == [event]


def test_streams_of_one_device(dev):
    """Of the pooled plans, the stream's own without a wait; another stream's
    with one."""
    f, _ = _graph()
    del f
    g, _ = _graph()
    assert dev.plans[1] is dev.plans[0] and not dev.streams[0].waits
    del g
    dev.streams[0] = Stream(0, 7)
    h, _ = _graph()
    assert dev.plans[2] is dev.plans[0] and len(dev.streams[0].waits) == 1


def test_plan_of_a_failed_forward_is_not_pooled(dev, monkeypatch):
    """What a failed call has left running is not covered by the plan's event."""
    plans = []

    def failing(mesh, x, u, f, lo, k, p, plan):
        plans.append(plan)
        raise _lib.PpmgError(-1, _lib.ERR_PART_UNASS, "particles lie in no sub")

    monkeypatch.setattr(core, "p2m", failing)
    with pytest.raises(_lib.PpmgError):
        _graph()
    assert plans[0].closed and not autograd._pool.get(0)


def test_failed_backward_is_covered(dev, monkeypatch):
    """The event covers what a failed adjoint launched."""
    f, xu = _graph()
    other = Stream(0, 9)

    def failing(*a, **k):
        dev.streams[0] = other
        raise _lib.PpmgError(-1, _lib.ERR_DEVICE, "failed")

    monkeypatch.setattr(core, "p2m_adjoint", failing)
    with pytest.raises(_lib.PpmgError):
        torch.autograd.grad(f.sum(), xu)
    del f
    assert autograd._pool[0][0][1].stream is other


def _pooled(dev):
    """Two plans in device 0's pool."""
    f, _ = _graph()
    g, _ = _graph()
    del f, g
    entries = list(autograd._pool[0])
    assert len(entries) == 2
    return [e[0] for e in entries]


def _once(real, error):
    """real, the first call of which raises error."""
    left = [error]

    def call(*a, **k):
        if left:
            raise left.pop()
        return real(*a, **k)
    return call


def test_given_back_when_the_field_does_not_fit(dev, monkeypatch):
    plans = _pooled(dev)
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", _once(torch.empty, torch.OutOfMemoryError("out of memory")))
        f, _ = _graph()
    assert f.shape == (8, 8, 1) and all(p.closed for p in plans)


@pytest.mark.parametrize("error", [torch.OutOfMemoryError("out of memory"),
                                   _lib.PpmgError(-1, _lib.ERR_ALLOC, "hipMalloc failed")])
def test_given_back_when_the_backward_does_not_fit(dev, monkeypatch, error):
    f, xu = _graph()
    plans = _pooled(dev)
    monkeypatch.setattr(core, "p2m_adjoint", _once(core.p2m_adjoint, error))
    torch.autograd.grad(f.sum(), xu)
    assert all(p.closed for p in plans) and not dev.plans[-1].closed


@pytest.mark.parametrize("error", [torch.OutOfMemoryError("out of memory"),
                                   _lib.PpmgError(-1, _lib.ERR_ALLOC, "hipMalloc failed")])
def test_out_of_memory_with_nothing_to_give_back(dev, monkeypatch, error):
    monkeypatch.setattr(core, "p2m", _once(core.p2m, error))
    with pytest.raises(type(error)):
        _graph()


def test_nothing_pooled_where_memory_is_short(dev, monkeypatch):
    """With less than SPARE_BYTES free, a graph's plan is freed with it, and
    so are those in the pool."""
    f, _ = _graph()
    plans = _pooled(dev)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d=None: (autograd.SPARE_BYTES - 1, 1 << 40))
    last = f.grad_fn.plan.plan
    del f
    assert last.closed and all(p.closed for p in plans) and not autograd._pool.get(0)


def test_free_memory_is_asked_for_now_and_then(dev, monkeypatch):
    """A steady loop does not ask at every graph, but does after ASK_SECONDS."""
    now, asked = [100.0], []
    monkeypatch.setattr(autograd, "_asked", {})
    monkeypatch.setattr(autograd.time, "monotonic", lambda: now[0])
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d=None: (asked.append(now[0]), (1 << 40, 1 << 40))[1])
    for _ in range(5):
        f, _ = _graph()
        del f
    assert len(asked) == 1
    now[0] += 2 * autograd.ASK_SECONDS
    for _ in range(5):
        f, _ = _graph()
        del f
    assert len(asked) == 2
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d=None: (0, 1 << 40))
    now[0] += 2 * autograd.ASK_SECONDS
    f, _ = _graph()
    del f
    assert not autograd._pool.get(0) and dev.plans[-1].closed
