"""torch.autograd wrapper of P2M on a fully periodic mesh (compact layout).

    field = p2m(xp, up, mesh, kernel=KERNEL_MP4, prec=PREC_F64)

field has shape (N_z, N_y, N_x, lda) (unique nodes).  The backward pass runs
the hand-written adjoint kernels (ppmg_p2m_adjoint): the strength gradient is
the M2P transpose of P2M, the position gradient uses the M'4 (or BSP2)
derivative stencil; both reuse the forward's sort permutation and cell keys
kept in the plan.

A plan's scratch is a dozen device allocations, which an optimisation loop
would make and free in every step (2.0 of 2.5 ms at 128^3, lda 3, on an
MI355X).  A graph's plan therefore goes back to a pool when the graph is
freed, and the next forward takes it from there, ordered after its last use
by an event.  The pool's memory is outside PyTorch's allocator, so it is kept
small and given back early: at most POOL_BYTES of scratch per device (a plan
over that, from about 390^3 cells on, is freed with its graph and made anew by
the next forward), none where less than SPARE_BYTES of the device is free when
a graph is freed, all of it when a forward or backward here runs out of memory,
and on release_plans(), for a client that is about to take nearly all there is.
"""
import sys
import threading

import torch

from . import core
from ._lib import ERR_ALLOC, KERNEL_MP4, PREC_F64, PpmgError

POOL_BYTES = 2 << 30
SPARE_BYTES = 16 << 30
_lock = threading.RLock()   # a collection inside it may run another plan's __del__
_pool = {}    # device index -> [(plan, event, (device, stream) of its last use, scratch bytes)]


def release_plans(device=None):
    """Frees the pooled plans of a device (all devices by default)."""
    with _lock:
        keys = list(_pool) if device is None else [torch.device("cuda", device).index]
        entries = [e for k in keys for e in _pool.pop(k, [])]
    for plan, event, _, _ in entries:
        event.synchronize()
        plan.close()


def _with_retry(call):
    """call(), again after giving the pool back if it runs out of memory."""
    try:
        return call()
    except (PpmgError, torch.OutOfMemoryError) as e:
        if (isinstance(e, PpmgError) and e.code != ERR_ALLOC) or not any(_pool.values()):
            raise
    release_plans()
    return call()


class _GraphPlan:
    """The plan of one forward, back in the pool when the graph lets go of it.
    Its scratch and work are those of the device and stream that are current
    (core._stream), whatever device the tensors are on: the plan is filed under
    that device, and a stream is told by its device too (every device's default
    stream has the handle 0)."""

    def __init__(self):
        self.device = torch.cuda.current_device()
        self.plan = self.event = self.last = None
        stream = torch.cuda.current_stream()
        here = (self.device, stream.cuda_stream)
        with _lock:
            free = _pool.get(self.device, [])
            # the most recently used one, of this stream where there is one
            at = next((i for i in reversed(range(len(free))) if free[i][2] == here), len(free) - 1)
            entry = free.pop(at) if free else None
        if entry is None:
            self.plan = core.Plan()
        else:
            self.plan, self.event, self.last, _ = entry
            if self.last != here:
                stream.wait_event(self.event)
        self.used()

    def used(self):
        """Marks the current stream's work so far as the plan's last use."""
        stream = torch.cuda.current_stream()
        here = (torch.cuda.current_device(), stream.cuda_stream)
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
            if torch.cuda.mem_get_info(self.device)[0] < SPARE_BYTES:   # (3 us)
                release_plans(self.device)
                self.drop()
                return
            n = self.plan.scratch_bytes()
            with _lock:
                free = _pool.setdefault(self.device, [])
                if n + sum(e[3] for e in free) <= POOL_BYTES:
                    free.append((self.plan, self.event, self.last, n))
                    self.plan = None
            if self.plan is not None:
                self.drop()
        except Exception:
            pass


class P2MFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, xp, up, mesh, kernel, prec):
        lda = up.shape[1]
        field = _with_retry(lambda: torch.empty(mesh.compact_shape(lda), dtype=core.VAL_DTYPE[prec], device=up.device))
        held = _GraphPlan()
        try:
            x, u = _with_retry(lambda: (xp.contiguous(), up.contiguous()))
            _with_retry(lambda: core.p2m(mesh, x, u, field, [0] * mesh.dim, kernel, prec, held.plan))
            held.used()
        except BaseException:
            held.drop()
            raise
        ctx.save_for_backward(xp, up)
        ctx.mesh, ctx.kernel, ctx.prec, ctx.plan = mesh, kernel, prec, held
        return field

    @staticmethod
    def backward(ctx, gfield):
        xp, up = ctx.saved_tensors
        want_x, want_u = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        if not (want_x or want_u):
            return None, None, None, None, None

        def adjoint():
            g = gfield.to(core.VAL_DTYPE[ctx.prec]).contiguous()
            gu, gx = core.p2m_adjoint(ctx.mesh, xp.contiguous(), up.contiguous(), g, [0] * ctx.mesh.dim,
                                      ctx.plan.plan, ctx.kernel, ctx.prec, want_u=want_u, want_x=want_x)
            return gu, gx if gx is None else gx.to(xp.dtype)

        try:
            gu, gx = _with_retry(adjoint)
        finally:
            ctx.plan.used()   # a failed call's launches too
        return gx, gu, None, None, None


def p2m(xp, up, mesh, kernel=KERNEL_MP4, prec=PREC_F64):
    if not mesh.periodic:
        raise ValueError("the autograd P2M needs a fully periodic mesh")
    return P2MFunction.apply(xp, up, mesh, kernel, prec)
