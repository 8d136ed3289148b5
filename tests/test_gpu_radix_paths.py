"""The radix sort of cell keys and the heads made from sorted keys, at the
sizes where their tiles and searches end."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def core():
    from ppm_legacy_amd import core as c
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return c


@pytest.mark.parametrize("n", [1, 63, 2047, 2048, 2049, 4096, 20001])
@pytest.mark.parametrize("cells", [(3, 2, 2), (16, 16, 14), (40, 33, 31), (130, 90, 60)])
@pytest.mark.parametrize("spread", ["inside", "some_outside", "one_cell"])
def test_rank_by_radix(core, monkeypatch, n, cells, spread):
    """util_rank by the radix sort against numpy's stable argsort: cell counts
    below and above the 4096-cell head tiles, 8- and 9-bit digits, particles in
    no box left out."""
    rng = np.random.default_rng(n + cells[0])
    x = rng.uniform(0, 1, (n, 3))
    if spread == "some_outside":
        x = x * 1.4 - 0.2
    elif spread == "one_cell":
        x = 0.5 + 1e-6 * x
    monkeypatch.setenv("PPMG_RADIX", "1")
    lpdx, lhbx = core.util_rank(torch.as_tensor(x).cuda(), [0.0] * 3, [1.0] * 3, cells, [1, 0, 0, 0, 1, 0])
    tot = np.array([cells[0] + 1, cells[1] + 1, cells[2]])
    i = np.floor(x * np.array(cells)).astype(int) + np.array([1, 0, 0])
    ok = ((i >= 0) & (i < tot)).all(1)
    key = i[:, 0] + tot[0] * (i[:, 1] + tot[1] * i[:, 2])
    at = np.nonzero(ok)[0]
    order = at[np.argsort(key[at], kind="stable")]
    assert np.array_equal(lpdx.cpu().numpy(), order + 1)
    want = np.concatenate([[0], np.cumsum(np.bincount(key[at], minlength=int(tot.prod())))]) + 1
    assert np.array_equal(lhbx.cpu().numpy(), want)


@pytest.mark.parametrize("dim", [2, 3])
def test_input_in_no_order(core, dim):
    """Large input in no order: the plan's second binning takes the radix sort;
    keys, permutation, heads and the field as the first binning's."""
    N = 1500 if dim == 2 else 130
    n = N ** dim
    assert n >= 1 << 21
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.rand((n, dim), dtype=torch.float64, device="cuda", generator=g)
    u = torch.randn((n, 1), dtype=torch.float64, device="cuda", generator=g)
    mesh = core.Mesh(dim, N + 1)
    plan = core.Plan()
    got = []
    for _ in range(3):
        f = torch.empty(mesh.compact_shape(1), dtype=torch.float64, device="cuda")
        core.p2m(mesh, x, u, f, [0] * dim, plan=plan)
        got.append((f,) + plan.sort_view())
    for a in got[1:]:
        for b, c in zip(a, got[0]):
            assert torch.equal(b, c)
    key, perm = got[0][1].long(), got[0][2].long()
    assert torch.equal(perm, torch.sort(key, stable=True)[1])
