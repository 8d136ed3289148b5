"""What a plan answers after a call that failed, or that replaced its binning."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MP4, BSP2 = 2, 1


@pytest.fixture(scope="module")
def core():
    from ppm_legacy_amd import core as c
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return c


def _forward(core, dim, kernel, N=12, n=700):
    """P2M of unordered particles into a stored box on a new plan (a slot
    table): mesh, positions, strengths, field, plan."""
    rng = np.random.default_rng(dim + 10 * kernel)
    mesh = core.Mesh(dim, N + 1)
    x = torch.as_tensor(rng.uniform(0, 1, (n, dim))).cuda()
    u = torch.as_tensor(rng.normal(size=(n, 2))).cuda()
    f = torch.zeros(mesh.padded_shape(2, [2] * dim), dtype=torch.float64, device="cuda")
    return mesh, x, u, f, core.p2m(mesh, x, u, f, [-2] * dim, kernel)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("kernel", [MP4, BSP2])
@pytest.mark.parametrize("where", ["ghost", "far"])
def test_adjoint_refused_after_m2p_with_particle_outside(core, dim, kernel, where):
    """M2P of as many particles, one of them outside the sub (on a ghost node,
    where the general path answers, or beyond the stored box, where it fails):
    the plan no longer holds the forward's binning, and the adjoint says so
    before any launch.  A new forward makes the plan good again."""
    from ppm_legacy_amd import _lib
    mesh, x, u, f, plan = _forward(core, dim, kernel)
    want = core.p2m_adjoint(mesh, x, u, f, [-2] * dim, plan, kernel)
    y = x.clone()
    y[5, 0] = 1.0 + 0.5 / 12 if where == "ghost" else 3.0
    out = torch.empty_like(u)
    if where == "ghost":
        core.m2p(mesh, y, f, [-2] * dim, out, kernel, plan=plan)
    else:
        with pytest.raises(_lib.PpmgError):
            core.m2p(mesh, y, f, [-2] * dim, out, kernel, plan=plan)
    with pytest.raises(_lib.PpmgError) as e:
        core.p2m_adjoint(mesh, x, u, f, [-2] * dim, plan, kernel)
    assert e.value.code == _lib.ERR_ARGUMENT
    g = f.clone()
    core.p2m(mesh, x, u, f, [-2] * dim, kernel, plan=plan)
    assert torch.equal(f, g)
    got = core.p2m_adjoint(mesh, x, u, f, [-2] * dim, plan, kernel)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_adjoint_after_m2p_without_binning(core, monkeypatch):
    """M2P on the general path bins nothing: the forward's binning stays."""
    mesh, x, u, f, plan = _forward(core, 3, MP4)
    want = core.p2m_adjoint(mesh, x, u, f, [-2] * 3, plan)
    monkeypatch.setenv("PPMG_GENERAL", "1")
    core.m2p(mesh, x, f, [-2] * 3, torch.empty_like(u), plan=plan)
    monkeypatch.delenv("PPMG_GENERAL")
    got = core.p2m_adjoint(mesh, x, u, f, [-2] * 3, plan)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def _refused(core, plan):
    """A call on `plan` whose scratch no device holds (its lda is 2^28, of
    which nothing is read: the allocation comes before any launch)."""
    import ctypes

    from ppm_legacy_amd import _lib
    mesh = core.Mesh(3, 9)
    field = torch.zeros(mesh.padded_shape(1, [2, 2, 2]), dtype=torch.float64, device="cuda")
    f = core.field_desc(mesh, field, [-2] * 3)
    f.lda = 1 << 28
    g = (ctypes.c_int * 3)(2, 2, 2)
    _lib.check(_lib.lib().ppmg_map_field_ghost(mesh.ref(), core.PREC_F64, ctypes.byref(f), g, _lib.MAP_GHOST_GET,
                                               plan.handle, None))


def test_refused_allocation_is_reported_once(core):
    """A device allocation that HIP itself refuses fails its own call and
    leaves nothing behind that a later call would report."""
    from ppm_legacy_amd import _lib
    plan = core.Plan()
    with pytest.raises(_lib.PpmgError) as e:
        _refused(core, plan)
    assert e.value.code == _lib.ERR_ALLOC
    mesh, x, u, f, plan = _forward(core, 3, MP4)
    assert abs(f[2:-3, 2:-3, 2:-3].sum().item() - u.sum().item()) < 1e-9 * u.abs().sum().item()


def test_graph_plan_retry_after_refused_allocation(core, monkeypatch):
    """A forward whose scratch HIP refuses gives the pooled plans back and
    runs again."""
    from ppm_legacy_amd import autograd
    mesh, x, u, _, _ = _forward(core, 3, MP4)
    autograd.release_plans()
    u.requires_grad_(True)
    want = autograd.p2m(x, u, mesh)
    keep = autograd.p2m(x, u, mesh)
    del keep                                   # its plan is in the pool
    real, calls = core.p2m, []

    def refusing(mesh_, x_, u_, f_, lo, kernel, prec, plan):
        calls.append(plan)
        if len(calls) == 1:
            autograd._pool.setdefault(0, []).append((core.Plan(), torch.cuda.Event(), 0, 0))
            _refused(core, plan)
        return real(mesh_, x_, u_, f_, lo, kernel, prec, plan)

    monkeypatch.setattr(core, "p2m", refusing)
    got = autograd.p2m(x, u, mesh)
    assert len(calls) == 2 and torch.equal(got, want)


def _crowded(core, N=128, n=1 << 19):
    """Particles in a quarter of the mesh per axis, 16 to a cell there."""
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.rand((n, 3), dtype=torch.float64, device="cuda", generator=g) / 4 + 0.4
    u = torch.randn((n, 1), dtype=torch.float64, device="cuda", generator=g)
    mesh = core.Mesh(3, N + 1)
    return mesh, x, u, torch.empty(mesh.compact_shape(1), dtype=torch.float64, device="cuda")


def test_work_list_without_memory(core, monkeypatch):
    """Crowded input with the work list's scratch refused (all else is there
    from calls of the general path): deposit, gather and adjoint run without
    it, bitwise as with it."""
    mesh, x, u, f = _crowded(core)

    def cycle(plan):
        core.p2m(mesh, x, u, f, [0] * 3, plan=plan)
        gu, gx = core.p2m_adjoint(mesh, x, u, f, [0] * 3, plan)
        out = torch.empty_like(u)
        core.m2p(mesh, x, f, [0] * 3, out, plan=plan)
        return f.clone(), gu, gx, out

    want = cycle(core.Plan())
    plan = core.Plan()
    monkeypatch.setenv("PPMG_GENERAL", "1")
    core.p2m(mesh, x, u, f, [0] * 3, plan=plan)
    core.p2m(mesh, x, u, f, [0] * 3, plan=plan)
    monkeypatch.delenv("PPMG_GENERAL")
    before = plan.scratch_bytes()
    monkeypatch.setenv("PPMG_FAIL_ALLOC_ABOVE", "0")
    got = cycle(plan)
    assert plan.scratch_bytes() == before
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    monkeypatch.delenv("PPMG_FAIL_ALLOC_ABOVE")
    got = cycle(plan)
    assert plan.scratch_bytes() > before       # the list has its scratch now
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_radix_binning_without_memory(core, monkeypatch):
    """Crowded input whose radix sort is refused its scratch is binned by
    counting: the same keys, permutation, heads and field."""
    mesh, x, u, f = _crowded(core)
    plan, got, size = core.Plan(), [], []
    # counted without the sort; sort refused, twice; sorted
    for env in ({"PPMG_RADIX": "0"}, {"PPMG_FAIL_ALLOC_ABOVE": "0"}, {"PPMG_FAIL_ALLOC_ABOVE": "0"}, {}):
        with monkeypatch.context() as m:
            for k, v in env.items():
                m.setenv(k, v)
            core.p2m(mesh, x, u, f, [0] * 3, plan=plan)
        size.append(plan.scratch_bytes())
        got.append((f.clone(),) + plan.sort_view())
    assert size[0] == size[1] == size[2] < size[3]
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(other, got[0]))


def test_rank_without_memory_for_the_sort(core, monkeypatch):
    """util_rank whose radix sort is refused its scratch ranks by counting."""
    g = torch.Generator(device="cuda").manual_seed(6)
    x = torch.rand((20000, 3), dtype=torch.float64, device="cuda", generator=g) * 1.1
    plan, got, size = core.Plan(), [], []
    for env in ({"PPMG_RADIX": "0"}, {"PPMG_RADIX": "1", "PPMG_FAIL_ALLOC_ABOVE": "0"}, {"PPMG_RADIX": "1"}):
        with monkeypatch.context() as m:
            for k, v in env.items():
                m.setenv(k, v)
            got.append(core.util_rank(x, [0.0] * 3, [1.0] * 3, (9, 8, 7), [1, 0, 0, 0, 1, 0], plan))
        size.append(plan.scratch_bytes())
    assert size[0] == size[1] < size[2]
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(other, got[0]))


@pytest.mark.parametrize("case", ["periodic", "open", "2d", "remesh", "m2p", "m2p_open"])
def test_slot_table_without_memory(core, monkeypatch, case):
    """A slot table (32 bytes a cell) that is refused: the particles are binned
    to heads and a permutation, with bitwise the same result."""
    dim, N, n = (2, 256, 3000) if case == "2d" else (3, 40, 3000)
    bc = [1] * (2 * dim)
    if "open" in case:
        bc[4:] = [7, 7]
    mesh = core.Mesh(dim, N + 1, bcdef=bc)
    rng = np.random.default_rng(12)
    x = torch.as_tensor(rng.uniform(0, 1, (n, dim))).cuda()
    u = torch.as_tensor(rng.normal(size=(n, 2))).cuda()
    f0 = torch.as_tensor(rng.normal(size=mesh.padded_shape(2, [2] * dim))).cuda()

    def run(plan):
        f, out = f0.clone(), torch.empty_like(u)
        if "m2p" in case:
            core.m2p(mesh, x, f, [-2] * dim, out, plan=plan)
            return out
        if case == "remesh":
            core.remesh(mesh, x, u, core.comp_weights(mesh, x), f, [-2] * dim, plan=plan)
        else:
            core.p2m(mesh, x, u, f, [-2] * dim, plan=plan)
        return f

    table = 32 * int(np.prod([N + (b != 1) for b in bc[::2]]))
    want, plan = run(core.Plan()), core.Plan()
    with monkeypatch.context() as m:
        m.setenv("PPMG_FAIL_ALLOC_ABOVE", str(table - 1))
        for _ in range(3):
            assert torch.equal(run(plan), want)
    assert plan.scratch_bytes() < table
    for _ in range(16):
        assert torch.equal(run(plan), want)
    assert plan.scratch_bytes() > table        # asked for again after 16 inputs


def test_registry_in_the_memory_of_one_plan(core, monkeypatch):
    """The registry keeps a plan per direction.  Where there is memory for one
    only, the idle one is given up; ppm_finalize gives up both.  A thread of its
    own, which starts with nothing."""
    import threading

    from ppm_legacy_amd import ppm
    N = 40
    rng = np.random.default_rng(13)
    x = torch.as_tensor(rng.uniform(0, 1, (3000, 3))).cuda()
    u = torch.as_tensor(rng.normal(size=(3000, 2))).cuda()
    mesh = core.Mesh(3, N + 1)
    f = torch.zeros(mesh.padded_shape(2, [2] * 3), dtype=torch.float64, device="cuda")
    back = torch.empty_like(u)
    p, q = core.p2m(mesh, x, u, f, [-2] * 3), core.m2p(mesh, x, f, [-2] * 3, back)
    one = max(p.scratch_bytes(), q.scratch_bytes())
    torch.cuda.synchronize()
    failed = []

    def work():
        try:
            assert ppm.ppm_init(3, ppm.ppm_kind_double, -15, None, 0) == 0
            info, topo, meshid = ppm.ppm_mktopo([0.0] * 3, [1.0] * 3, [1] * 6, [N + 1] * 3, [2] * 3)
            assert info == 0
            monkeypatch.setenv("PPMG_FAIL_ALLOC_TOTAL", str(one + 65536))
            for _ in range(2):
                g, b = torch.zeros_like(f), torch.zeros_like(u)
                torch.cuda.synchronize()
                assert ppm.ppm_interp_m2p(x, 3000, b, topo, meshid, MP4, [2] * 3, f) == 0
                assert ppm.ppm_interp_p2m(x, 3000, u, topo, meshid, MP4, [2] * 3, g) == 0
                assert torch.equal(g, f) and torch.equal(b, back)
            assert ppm.ppm_finalize() == 0
            core.p2m(mesh, x, u, g, [-2] * 3)
            torch.cuda.synchronize()
            assert torch.equal(g, f)
        except BaseException as e:
            failed.append(repr(e))

    t = threading.Thread(target=work)
    t.start()
    t.join()
    assert not failed


@pytest.mark.parametrize("sizes", [(12,), (4, 30)], ids=["new", "grown"])
def test_sort_view_after_a_refused_binning(core, sizes):
    """Particles outside the sub: P2M refuses them, and the plan's view still
    has arrays of the right size, with the keys (-1 outside)."""
    from ppm_legacy_amd import _lib
    plan = core.Plan()
    for N in sizes:
        rng = np.random.default_rng(N)
        n = N ** 3
        x = rng.uniform(0, 1, (n, 3))
        x[[1, n // 2]] = [1.5, 0.5, 0.5]
        mesh = core.Mesh(3, N + 1)
        u = torch.ones((n, 1), dtype=torch.float64, device="cuda")
        f = torch.empty(mesh.compact_shape(1), dtype=torch.float64, device="cuda")
        if N != sizes[-1]:       # a smaller binning first, which leaves small arrays
            core.p2m(mesh, torch.as_tensor(rng.uniform(0, 1, (n, 3))).cuda(), u, f, [0] * 3, plan=plan)
            plan.sort_view()
            continue
        xd = torch.as_tensor(x).cuda()
        with pytest.raises(_lib.PpmgError) as e:
            core.p2m(mesh, xd, u, f, [0] * 3, plan=plan)
        assert e.value.code == _lib.ERR_PART_UNASS
        key, perm, start = plan.sort_view()
        c = np.floor(x * N).astype(int)
        want = np.where((x < 1).all(1), c[:, 0] + N * (c[:, 1] + N * c[:, 2]), -1)
        assert np.array_equal(key.cpu().numpy(), want)
        assert perm.shape == (n,) and start.shape == (N ** 3 + 1,)
        xd[[1, n // 2]] = 0.5
        core.p2m(mesh, xd, u, f, [0] * 3, plan=plan)
        assert abs(f.sum().item() - n) < 1e-9 * n
