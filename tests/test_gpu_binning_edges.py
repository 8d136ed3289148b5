"""Binning forms at the sizes where their digits, tiles and tables end."""
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


@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, 8191, 8192, 8193, 30001])
@pytest.mark.parametrize("cells,bits", [((8, 7, 6), 9), ((50, 40, 36), 17), ((64, 50, 40), 18), ((16, 16, 14), 12)])
@pytest.mark.parametrize("outside", [False, True])
def test_rank_radix_digits(core, monkeypatch, n, cells, bits, outside):
    """util_rank by radix passes of 9 bits (keys of 9, 17 and 18) and of 8,
    around their tiles of 8192 and 4096 pairs, with particles in no box left
    out (the values past the last box not written): numpy's stable argsort."""
    ngl = [1, 0, 0, 0, 1, 0]
    tot = np.array(cells) + np.array(ngl[:3]) + np.array(ngl[3:])
    assert int(np.prod(tot)).bit_length() == bits      # keys 0 .. prod(tot)
    rng = np.random.default_rng(n + bits)
    x = rng.uniform(0, 1, (n, 3))
    if outside:
        x = x * 1.4 - 0.2
    monkeypatch.setenv("PPMG_RADIX", "1")
    lpdx, lhbx = core.util_rank(torch.as_tensor(x).cuda(), [0.0] * 3, [1.0] * 3, cells, ngl)
    i = np.floor(x * np.array(cells)).astype(int) + np.array(ngl[:3])
    ok = ((i >= 0) & (i < tot)).all(1)
    key = i[:, 0] + tot[0] * (i[:, 1] + tot[1] * i[:, 2])
    at = np.nonzero(ok)[0]
    assert np.array_equal(lpdx.cpu().numpy(), at[np.argsort(key[at], kind="stable")] + 1)
    want = np.concatenate([[0], np.cumsum(np.bincount(key[at], minlength=int(tot.prod())))]) + 1
    assert np.array_equal(lhbx.cpu().numpy(), want)


@pytest.mark.parametrize("shape", [(5, 6, 4), (16, 22, 13), (33, 25, 18)])
@pytest.mark.parametrize("bc", [[1, 1, 1, 1, 2, 2], [2, 2, 1, 1, 1, 1], [2] * 6], ids=["open_z", "open_x", "open"])
@pytest.mark.parametrize("kernel", [MP4, BSP2])
@pytest.mark.parametrize("prec", [F64, F32C, F32])
def test_deposit_on_open_axes_accepts_the_faces(core, monkeypatch, shape, bc, kernel, prec):
    """Unordered particles, some on the open faces: every one is in the sub, so
    the deposit answers on the slot table, on heads (bitwise) and on the general
    path (1e-13 of the maximum in FP64, FP32 forms 2e-5: sums of up to a few
    hundred terms)."""
    rng = np.random.default_rng(shape[0] + kernel)
    n = int(np.prod(shape)) + 40
    x = rng.uniform(0, 0.999, (n, 3))
    for d in range(3):
        x[10 * d:10 * d + 5, d] = 0.0
        if bc[2 * d] == 2:
            x[10 * d + 5:10 * d + 10, d] = 1.0
    mesh = core.Mesh(3, [v + 1 for v in shape], None, None, bc)
    vdt = core.VAL_DTYPE[prec]
    xd = torch.as_tensor(x).to(core.POS_DTYPE[prec]).cuda()
    u = torch.as_tensor(rng.normal(size=(n, 3))).to(vdt).cuda()

    def run():
        f = torch.full(mesh.padded_shape(3, [2] * 3), 7.0, dtype=vdt, device="cuda")
        core.p2m(mesh, xd, u, f, [-2] * 3, kernel, prec)
        return f

    f = run()
    monkeypatch.setenv("PPMG_NO_TABLE", "1")
    assert torch.equal(run(), f)
    monkeypatch.delenv("PPMG_NO_TABLE")
    monkeypatch.setenv("PPMG_GENERAL", "1")
    ref = run()
    assert ((f - ref).abs().max() / ref.abs().max()).item() < (1e-13 if prec == F64 else 2e-5)
