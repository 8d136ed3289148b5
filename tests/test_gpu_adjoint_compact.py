"""The compact-layout adjoint (2D, and BSP2 in 3D) against the general one."""
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


def _compare(core, monkeypatch, shape, kernel, prec, lda, lo, seed):
    dim = len(shape)
    rng = np.random.default_rng(seed)
    n = int(np.prod(shape))
    x = np.concatenate([rng.uniform(0, 0.9999, (n + 3, dim)), 0.5 + 0.02 * rng.uniform(0, 1, (40, dim))])
    side = np.array(shape) / max(shape)
    mesh = core.Mesh(dim, [v + 1 for v in shape], [0.0] * dim, list(side))
    pdt, vdt = core.POS_DTYPE[prec], core.VAL_DTYPE[prec]
    xd = torch.as_tensor(x * side).to(pdt).cuda()
    u = torch.as_tensor(rng.normal(size=(len(x), lda))).to(vdt).cuda()
    fs = mesh.compact_shape(lda) if lo == 0 else mesh.padded_shape(lda, [-lo] * dim)
    g = torch.as_tensor(rng.normal(size=fs)).to(vdt).cuda()

    def run():
        f = torch.empty(fs, dtype=vdt, device="cuda")
        plan = core.p2m(mesh, xd, u, f, [lo] * dim, kernel, prec)
        return core.p2m_adjoint(mesh, xd, u, g, [lo] * dim, plan, kernel, prec)

    got = run()
    monkeypatch.setenv("PPMG_NO_TABLE", "1")     # cell order instead of the caller's: the same sums
    for a, b in zip(run(), got):
        assert torch.equal(a, b)
    monkeypatch.delenv("PPMG_NO_TABLE")
    monkeypatch.setenv("PPMG_GENERAL", "1")
    ref = run()
    monkeypatch.delenv("PPMG_GENERAL")
    if prec == F32C and lo == 0:     # the same sums in the same order: the same bits
        for a, b in zip(got, ref):
            assert torch.equal(a, b)
    # (FP64 products may fuse differently: 8 to 16 terms each, 1e-13 of the
    # maximum; the FP32 form 2e-5)
    for a, b in zip(got, ref):
        assert ((a - b).abs().max() / b.abs().max()).item() < (1e-13 if prec == F64 else 2e-5)


@pytest.mark.parametrize("shape", [(4, 4), (5, 13), (16, 15), (17, 30), (301, 40)])
@pytest.mark.parametrize("kernel", [MP4, BSP2])
@pytest.mark.parametrize("prec", [F64, F32C, F32])
@pytest.mark.parametrize("lda", [1, 2, 4, 5])
def test_adjoint_2d(core, monkeypatch, shape, kernel, prec, lda):
    _compare(core, monkeypatch, shape, kernel, prec, lda, 0, shape[0] + lda)


@pytest.mark.parametrize("shape", [(4, 4, 4), (15, 16, 9), (16, 17, 33), (33, 31, 20)])
@pytest.mark.parametrize("prec", [F64, F32C, F32])
@pytest.mark.parametrize("lda", [1, 3, 4])
@pytest.mark.parametrize("lo", [0, -1, -2])
def test_adjoint_3d_bsp2(core, monkeypatch, shape, prec, lda, lo):
    _compare(core, monkeypatch, shape, BSP2, prec, lda, lo, shape[0] + lda)
