"""torch.autograd wrapper of P2M on a fully periodic mesh (compact layout).

    field = p2m(xp, up, mesh, kernel=KERNEL_MP4, prec=PREC_F64)

field has shape (N_z, N_y, N_x, lda) (unique nodes).  The backward pass runs
the hand-written adjoint kernels (ppmg_p2m_adjoint): the strength gradient is
the M2P transpose of P2M, the position gradient uses the M'4 (or BSP2)
derivative stencil.  The 3D M'4 adjoint reads the forward's binning, kept in the
plan; the 2D and BSP2 ones take each particle's cell from its position (in the
forward's order where it left a permutation).

A plan's scratch is a dozen device allocations, which an optimisation loop
would make and free in every step (2.0 of 2.5 ms at 128^3, lda 3, on an
MI355X).  A graph's plan therefore goes back to a pool when the graph is
freed, and the next forward takes it from there, ordered after its last use
by an event.  The pool's memory is outside PyTorch's allocator, so it is kept
small and given back early: at most POOL_BYTES of scratch per device (a plan
over that, from about 390^3 cells on, is freed with its graph and made anew by
the next forward), none where less than SPARE_BYTES of the device is free when
a graph is freed (a steady loop asks every ASK_SECONDS), all of it when a forward
or backward here runs out of memory, and on release_plans(), for a client that
is about to take nearly all there is.
"""
import sys
import threading
import time

import torch

from . import core
from ._lib import ERR_ALLOC, KERNEL_MP4, PREC_F64, PpmgError

POOL_BYTES = 2 << 30
SPARE_BYTES = 16 << 30
ASK_SECONDS = 0.1
_lock = threading.RLock()   # a collection inside it may run another plan's __del__
_asked = {}   # device index -> when its free memory was last asked for
_pool = {}    # device index -> [(plan, event, (device, stream) of its last use, scratch bytes)]


def release_plans(device=None):
    """Frees the pooled plans of a device (all devices by default)."""
    with _lock:
        keys = list(_pool) if device is None else [torch.device("cuda", device).index]
        entries = [e for k in keys for e in _pool.pop(k, [])]
    for plan, event, _, _ in entries:
        event.synchronize()
        plan.close()


def _given_back(e):
    """Whether e says that memory ran out and the pool had some to give back:
    worth another try."""
    with _lock:
        some = any(_pool.values())
    if not some or (isinstance(e, PpmgError) and e.code != ERR_ALLOC):
        return False
    release_plans()
    return True


class _GraphPlan:
    """The plan of one forward, back in the pool when the graph lets go of it.
    Its scratch and work are those of the device and stream that are current
    (core._stream), whatever device the tensors are on: the plan is filed under
    that device, and a stream is told by its device too (every device's default
    stream has the handle 0)."""

    def __init__(self):
        stream = torch.cuda.current_stream()
        here = (stream.device_index, stream.cuda_stream)
        self.device = stream.device_index
        self.plan = self.event = self.last = None
        self.pooled = -1          # the plan's scratch as it lay in the pool
        with _lock:
            free = _pool.get(self.device)
            if free:
                # the most recently used one, of this stream where there is one
                at = next((i for i in reversed(range(len(free))) if free[i][2] == here), -1)
                self.plan, self.event, self.last, self.pooled = free.pop(at)
        if self.plan is None:
            self.plan = core.Plan()
        elif self.last != here:
            stream.wait_event(self.event)

    def used(self):
        """Marks the current stream's work so far as the plan's last use."""
        stream = torch.cuda.current_stream()
        here = (stream.device_index, stream.cuda_stream)
        if self.event is None or self.last[0] != here[0]:   # an event belongs to one device
            self.event = torch.cuda.Event()
        self.event.record(stream)
        self.last = here

    def drop(self):
        """Frees the plan: a failed call may have left work running that no
        event covers (freeing device memory waits for it)."""
        plan, self.plan = self.plan, None
        plan.close()

    def __del__(self):
        if self.plan is None or sys.is_finalizing():
            return
        try:
            if self.event is None:     # never used
                return self.drop()
            n, now = self.plan.scratch_bytes(), time.monotonic()
            # asking for the free memory takes up to 18 us (of 140 for a small
            # mesh's step): for a plan that is new to the pool, else now and then
            if n != self.pooled or now - _asked.get(self.device, 0.0) > ASK_SECONDS:
                _asked[self.device] = now
                if torch.cuda.mem_get_info(self.device)[0] < SPARE_BYTES:
                    release_plans(self.device)
                    return self.drop()
            with _lock:
                free = _pool.setdefault(self.device, [])
                if n + sum(e[3] for e in free) <= POOL_BYTES:
                    free.append((self.plan, self.event, self.last, n))
                    self.plan = None
            if self.plan is not None:
                self.drop()
        except Exception:
            pass


def _forward(xp, up, mesh, kernel, prec):
    field = torch.empty(mesh.compact_shape(up.shape[1]), dtype=core.VAL_DTYPE[prec], device=up.device)
    held = _GraphPlan()
    try:
        core.p2m(mesh, xp.contiguous(), up.contiguous(), field, [0] * mesh.dim, kernel, prec, held.plan)
        held.used()
    except BaseException:
        held.drop()
        raise
    return field, held


def _backward(ctx, gfield):
    xp, up = ctx.saved_tensors
    g = gfield.to(core.VAL_DTYPE[ctx.prec]).contiguous()
    try:
        gu, gx = core.p2m_adjoint(ctx.mesh, xp.contiguous(), up.contiguous(), g, [0] * ctx.mesh.dim, ctx.plan.plan,
                                  ctx.kernel, ctx.prec, want_u=ctx.needs_input_grad[1], want_x=ctx.needs_input_grad[0])
    finally:
        ctx.plan.used()   # a failed call's launches too
    return gx if gx is None else gx.to(xp.dtype), gu, None, None, None


class P2MFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, xp, up, mesh, kernel, prec):
        try:
            field, held = _forward(xp, up, mesh, kernel, prec)
        except (PpmgError, torch.OutOfMemoryError) as e:
            if not _given_back(e):
                raise
            field, held = _forward(xp, up, mesh, kernel, prec)
        ctx.save_for_backward(xp, up)
        ctx.mesh, ctx.kernel, ctx.prec, ctx.plan = mesh, kernel, prec, held
        return field

    @staticmethod
    def backward(ctx, gfield):
        if not (ctx.needs_input_grad[0] or ctx.needs_input_grad[1]):
            return None, None, None, None, None
        try:
            return _backward(ctx, gfield)
        except (PpmgError, torch.OutOfMemoryError) as e:
            if not _given_back(e):
                raise
            return _backward(ctx, gfield)


def p2m(xp, up, mesh, kernel=KERNEL_MP4, prec=PREC_F64):
    if not mesh.periodic:
        raise ValueError("the autograd P2M needs a fully periodic mesh")
    return P2MFunction.apply(xp, up, mesh, kernel, prec)
