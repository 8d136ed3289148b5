"""Weight tables of more particles than one launch takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_comp_weights_over_2_31_particles():
    """2D, M'4, FP32: 2^31 + 5 particles (86 GB with the tables), two lanes
    each.  The rows at both ends and around the launches' seams equal those of
    a small call, bit for bit."""
    from ppm_legacy_amd import core
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    torch.cuda.empty_cache()
    n, w = (1 << 31) + 5, 300
    mesh = core.Mesh(2, 65)
    x = torch.empty((n, 2), dtype=torch.float32, device="cuda").fill_(0.37)
    g = torch.Generator(device="cuda").manual_seed(2)
    rows = [slice(0, w), slice((1 << 30) - w, (1 << 30) + w), slice((1 << 31) - w, n)]
    for r in rows:
        x[r] = torch.rand((r.stop - r.start, 2), dtype=torch.float32, device="cuda", generator=g)
    big = core.comp_weights(mesh, x, prec=core.PREC_F32)
    try:
        for r in rows:
            small = core.comp_weights(mesh, x[r].contiguous(), prec=core.PREC_F32)
            assert all(torch.equal(a[r], b) for a, b in zip(big, small))
    finally:
        del x, big
        torch.cuda.empty_cache()
