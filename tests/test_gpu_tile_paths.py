"""The tiled kernels at the occupancies and sizes where they change path."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MP4, BSP2 = 2, 1
F64, F32C, F32 = 0, 1, 2


@pytest.fixture(scope="module")
def core():
    from ppm_legacy_amd import core as c
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return c


def _general(monkeypatch, call):
    monkeypatch.setenv("PPMG_GENERAL", "1")
    r = call()
    monkeypatch.delenv("PPMG_GENERAL")
    return r


@pytest.mark.parametrize("extra", [0, 1, 4, 14, 15, 16, 17, 64])
@pytest.mark.parametrize("kernel", [MP4, BSP2])
@pytest.mark.parametrize("lda", [1, 3, 4])
def test_deposit_second_particles(core, monkeypatch, extra, kernel, lda):
    """One particle per cell and a second (every fifth of those a third) in
    `extra` cells of one 16 x 4 block: around the number of second particles
    the deposit stages.  FP64 sums of at most 100 terms against the general
    path: 1e-13 of the maximum; both binning forms bitwise the same."""
    N = 24
    rng = np.random.default_rng(extra + 100 * lda)
    i = np.arange(N ** 3)
    cells = np.stack([i % N, (i // N) % N, i // N ** 2], 1)
    block = np.stack([np.arange(extra) % 16 + 3, np.arange(extra) // 16 + 6, np.full(extra, 11)], 1)
    cells = np.concatenate([cells, block, block[::5]]).astype(float)
    x = (cells + rng.uniform(0.02, 0.98, cells.shape)) / N
    order = rng.permutation(len(x))
    mesh = core.Mesh(3, N + 1)
    xd = torch.as_tensor(x[order]).cuda()
    u = torch.as_tensor(rng.normal(size=(len(x), lda))).cuda()

    def p2m():
        f = torch.empty(mesh.compact_shape(lda), dtype=torch.float64, device="cuda")
        core.p2m(mesh, xd, u, f, [0] * 3, kernel)
        return f

    f, ref = p2m(), _general(monkeypatch, p2m)
    assert ((f - ref).abs().max() / ref.abs().max()).item() < 1e-13
    monkeypatch.setenv("PPMG_NO_TABLE", "1")
    assert torch.equal(f, p2m())


@pytest.mark.parametrize("N", [4, 7, 16, 31, 33])
@pytest.mark.parametrize("prec", [F64, F32C, F32])
def test_small_meshes_short_chunks(core, monkeypatch, N, prec):
    """Meshes of one to a few planes per workgroup: deposit, gather and adjoint
    against the general path (1e-13 in FP64; FP32 forms 2e-5 of the maximum)."""
    rng = np.random.default_rng(N)
    n = N ** 3 + 5
    mesh = core.Mesh(3, N + 1)
    pdt, vdt = core.POS_DTYPE[prec], core.VAL_DTYPE[prec]
    x = torch.as_tensor(rng.uniform(0, 0.9999, (n, 3))).to(pdt).cuda()
    u = torch.as_tensor(rng.normal(size=(n, 3))).to(vdt).cuda()
    g = torch.as_tensor(rng.normal(size=mesh.compact_shape(3))).to(vdt).cuda()

    def run():
        f = torch.empty(mesh.compact_shape(3), dtype=vdt, device="cuda")
        plan = core.p2m(mesh, x, u, f, [0] * 3, MP4, prec)
        gu, gx = core.p2m_adjoint(mesh, x, u, g, [0] * 3, plan, MP4, prec)
        out = torch.empty_like(u)
        core.m2p(mesh, x, g, [0] * 3, out, MP4, prec)
        return f, gu, gx, out

    tol = 1e-13 if prec == F64 else 2e-5
    for a, b in zip(run(), _general(monkeypatch, run)):
        assert ((a - b).abs().max() / b.abs().max()).item() < tol


@pytest.mark.parametrize("shape", [(40, 36, 70), (16, 21, 5), (15, 60, 33)])
@pytest.mark.parametrize("bc", [[1] * 6, [1, 1, 1, 1, 2, 2], [2] * 6], ids=["periodic", "open_z", "open"])
@pytest.mark.parametrize("kernel", [MP4, BSP2])
def test_crowded_work_list(core, monkeypatch, shape, bc, kernel):
    """Crowded cells (up to hundreds of particles) beside empty space, so that
    tile columns are cut into pieces of every length; ragged tiles and segment
    ends.  Deposit, gather and adjoint against the general path (sums of up to
    a few thousand terms in FP64: 1e-12 of the maximum); the plan's second and
    third pass (radix binning) bitwise like its first."""
    rng = np.random.default_rng(shape[2] + kernel)
    x = np.concatenate([rng.normal(0.45, 0.03, (5000, 3)).clip(0.01, 0.99), rng.uniform(0, 0.999, (3000, 3))])
    side = np.array(shape) / max(shape)
    mesh = core.Mesh(3, [n + 1 for n in shape], [0.0] * 3, list(side), bc)
    xd = torch.as_tensor(x * side).cuda()
    u = torch.as_tensor(rng.normal(size=(len(x), 3))).cuda()
    fs, lo = mesh.padded_shape(3, [2] * 3), [-2] * 3
    g = torch.as_tensor(rng.normal(size=fs)).cuda()
    pp, pm = core.Plan(), core.Plan()

    def run(pp=None, pm=None):
        f = torch.empty(fs, dtype=torch.float64, device="cuda")
        pp = core.p2m(mesh, xd, u, f, lo, kernel, plan=pp)
        gu, gx = core.p2m_adjoint(mesh, xd, u, g, lo, pp, kernel)
        out = torch.empty_like(u)
        core.m2p(mesh, xd, g, lo, out, kernel, plan=pm)
        return f, gu, gx, out

    first = run(pp, pm)
    for _ in range(2):
        for a, b in zip(run(pp, pm), first):
            assert torch.equal(a, b)
    for a, b in zip(first, _general(monkeypatch, run)):
        assert ((a - b).abs().max() / b.abs().max()).item() < 1e-12


@pytest.mark.parametrize("nx", [27, 29, 55, 58])
@pytest.mark.parametrize("bc", [[1] * 6, [1, 1, 1, 1, 2, 2], [2] * 6], ids=["periodic", "open_z", "open"])
@pytest.mark.parametrize("parts", ["lattice", "random", "blob"])
@pytest.mark.parametrize("prec", [F64, F32C])
def test_gather_wide_rows(core, monkeypatch, nx, bc, parts, prec):
    """Meshes whose M'4 gather takes rows of 32 lanes (29 cells to a tile), on
    every binning form: bitwise the same on all three passes of a plan, and
    against the general path (64 terms: 1e-13 of the maximum in FP64, FP32c
    with FP64 sums of FP32 nodes 1e-6)."""
    shape = (nx, 19, 10)
    rng = np.random.default_rng(nx)
    if parts == "lattice":
        i = np.arange(nx * 19 * 10)
        x = (np.stack([i % nx, (i // nx) % 19, i // (nx * 19)], 1) + rng.uniform(0.05, 0.95, (len(i), 3))) / shape
    elif parts == "random":
        x = rng.uniform(0, 0.999, (nx * 190, 3))
    else:
        x = np.concatenate([rng.normal(0.5, 0.04, (4000, 3)).clip(0.01, 0.99), rng.uniform(0, 0.999, (500, 3))])
    side = np.array(shape) / nx
    mesh = core.Mesh(3, [n + 1 for n in shape], [0.0] * 3, list(side), bc)
    xd = torch.as_tensor(x * side).to(core.POS_DTYPE[prec]).cuda()
    vdt = core.VAL_DTYPE[prec]
    for lda in (1, 3, 4):
        f = torch.as_tensor(rng.normal(size=mesh.padded_shape(lda, [2] * 3))).to(vdt).cuda()

        def m2p(plan=None):
            out = torch.empty((len(x), lda), dtype=vdt, device="cuda")
            core.m2p(mesh, xd, f, [-2] * 3, out, MP4, prec, plan=plan)
            return out

        plan = core.Plan()
        got = m2p(plan)
        for _ in range(2):
            assert torch.equal(got, m2p(plan))
        ref = _general(monkeypatch, m2p)
        assert ((got - ref).abs().max() / ref.abs().max()).item() < (1e-13 if prec == F64 else 1e-6)


@pytest.mark.parametrize("shape", [(4, 5), (30, 17), (65, 40)])
@pytest.mark.parametrize("ghost", [0, 2])
@pytest.mark.parametrize("kernel", [MP4, BSP2])
@pytest.mark.parametrize("prec", [F64, F32])
def test_plane_lattice_without_binning(core, shape, ghost, kernel, prec):
    """2D: a plan that has seen a lattice in cell order gathers at the next one
    without a binning pass.  One plan is fed the lattice (binned), two more
    (no pass), one with two particles swapped and one with a NaN (checked, then
    binned again), and a lattice after 16 binned ones: every output, or error,
    is bitwise that of a fresh plan, and sort_view gives the identity."""
    nx, ny = shape
    n = nx * ny
    rng = np.random.default_rng(nx + ghost)
    i = np.arange(n)
    side = np.array(shape) / max(shape)
    mesh = core.Mesh(2, [nx + 1, ny + 1], [0.0] * 2, list(side))
    vdt = core.VAL_DTYPE[prec]
    fs = mesh.padded_shape(3, [ghost] * 2) if ghost else mesh.compact_shape(3)
    f = torch.as_tensor(rng.normal(size=fs)).to(vdt).cuda()

    def call(x, plan=None):
        out = torch.zeros((n, 3), dtype=vdt, device="cuda")
        try:
            core.m2p(mesh, x, f, [-ghost] * 2, out, kernel, prec, plan=plan)
        except RuntimeError as e:
            return str(e)
        return out

    def lattice():
        x = (np.stack([i % nx, i // nx], 1) + rng.uniform(0.05, 0.95, (n, 2))) / shape * side
        return torch.as_tensor(x).to(core.POS_DTYPE[prec]).cuda()

    plan = core.Plan()
    for case in ["lattice"] * 3 + ["swapped", "lattice", "lattice"] + ["lattice"] * 16 + ["nan", "lattice"]:
        x = lattice()
        if case == "swapped":
            x[[0, n - 1]] = x[[n - 1, 0]]
        elif case == "nan":
            x[n // 2, 1] = float("nan")
        got, ref = call(x, plan), call(x)
        assert type(got) is type(ref), case
        if isinstance(ref, str):
            assert got == ref
            continue
        assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(ref)), case
        if case == "lattice":
            k, perm, start = plan.sort_view()
            assert np.array_equal(start.cpu().numpy(), np.arange(n + 1))
            assert np.array_equal(perm.cpu().numpy(), np.arange(n))
            assert np.array_equal(k.cpu().numpy(), np.arange(n))


@pytest.mark.parametrize("shape", [(5, 6, 4), (16, 22, 13), (33, 25, 18)])
@pytest.mark.parametrize("bc", [[1, 1, 1, 1, 2, 2], [2, 2, 1, 1, 1, 1], [2] * 6], ids=["open_z", "open_x", "open"])
@pytest.mark.parametrize("kernel", [MP4, BSP2])
@pytest.mark.parametrize("prec", [F64, F32C, F32])
def test_slot_table_on_open_axes(core, monkeypatch, shape, bc, kernel, prec):
    """Unordered particles on a mesh with open axes, some on its faces: deposit
    and gather on the slot table bitwise as on heads and permutation, and
    against the general path (sums of up to a few hundred terms: 1e-13 of the
    maximum in FP64, FP32 forms 2e-5)."""
    rng = np.random.default_rng(shape[0] + kernel)
    n = int(np.prod(shape)) + 40
    x = rng.uniform(0, 0.999, (n, 3))
    for d in range(3):
        x[10 * d:10 * d + 5, d] = 0.0
        if bc[2 * d] == 2:
            x[10 * d + 5:10 * d + 10, d] = 1.0
    side = np.array(shape) / max(shape)
    mesh = core.Mesh(3, [v + 1 for v in shape], [0.0] * 3, list(side), bc)
    vdt = core.VAL_DTYPE[prec]
    xd = torch.as_tensor(x).to(core.POS_DTYPE[prec]) * torch.as_tensor(side).to(core.POS_DTYPE[prec])
    xd = torch.minimum(xd, torch.as_tensor(mesh.max_phys).to(xd.dtype)).cuda()
    u = torch.as_tensor(rng.normal(size=(n, 3))).to(vdt).cuda()
    g = torch.as_tensor(rng.normal(size=mesh.padded_shape(3, [2] * 3))).to(vdt).cuda()

    def run():
        f = torch.empty_like(g)
        try:
            core.p2m(mesh, xd, u, f, [-2] * 3, kernel, prec)
        except RuntimeError as e:      # faces the sub does not hold: the same error on every path
            f = torch.full((1,), float(hash(str(e)) % 1000 + 1), dtype=vdt, device="cuda")
        out = torch.empty_like(u)
        core.m2p(mesh, xd, g, [-2] * 3, out, kernel, prec)
        return f, out

    got = run()
    monkeypatch.setenv("PPMG_NO_TABLE", "1")
    for a, b in zip(run(), got):
        assert torch.equal(a, b)
    monkeypatch.delenv("PPMG_NO_TABLE")
    for a, b in zip(got, _general(monkeypatch, run)):
        assert ((a - b).abs().max() / b.abs().max()).item() < (1e-13 if prec == F64 else 2e-5)


@pytest.mark.parametrize("nx", [27, 29, 55, 58])
@pytest.mark.parametrize("ghost", [0, 2])
@pytest.mark.parametrize("prec", [F64, F32C])
def test_adjoint_wide_rows(core, monkeypatch, nx, ghost, prec):
    """Meshes whose M'4 adjoint takes rows of 32 lanes, on the slot table and on
    heads (bitwise the same), and against the general path (64 terms: 1e-13 of
    the maximum in FP64; FP32c 2e-5)."""
    shape = (nx, 19, 10)
    rng = np.random.default_rng(nx + ghost)
    x = np.concatenate([rng.uniform(0, 0.999, (nx * 190, 3)), 0.5 + 0.03 * rng.uniform(0, 1, (6, 3))])
    side = np.array(shape) / nx
    mesh = core.Mesh(3, [n + 1 for n in shape], [0.0] * 3, list(side))
    vdt = core.VAL_DTYPE[prec]
    xd = torch.as_tensor(x * side).to(core.POS_DTYPE[prec]).cuda()
    for lda in (1, 3, 4):
        u = torch.as_tensor(rng.normal(size=(len(x), lda))).to(vdt).cuda()
        fs = mesh.padded_shape(lda, [ghost] * 3) if ghost else mesh.compact_shape(lda)
        g = torch.as_tensor(rng.normal(size=fs)).to(vdt).cuda()

        def run():
            f = torch.empty_like(g)
            plan = core.p2m(mesh, xd, u, f, [-ghost] * 3, MP4, prec)
            return core.p2m_adjoint(mesh, xd, u, g, [-ghost] * 3, plan, MP4, prec)

        got = run()
        monkeypatch.setenv("PPMG_NO_TABLE", "1")
        for a, b in zip(run(), got):
            assert torch.equal(a, b)
        monkeypatch.delenv("PPMG_NO_TABLE")
        for a, b in zip(got, _general(monkeypatch, run)):
            assert ((a - b).abs().max() / b.abs().max()).item() < (1e-13 if prec == F64 else 2e-5)
