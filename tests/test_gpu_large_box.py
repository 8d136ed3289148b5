"""Stored boxes of more nodes than 32 bits count."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unordered", [True, False])
def test_ghost_shell_over_2_32_nodes(unordered):
    """8^3 cells in a box with 12.7 million ghost planes on either side in z
    (4.29e9 nodes, 17 GB in FP32; the planes' count is just over 2^32 nodes, so
    that a product in 32 bits would be small): the nodes near the mesh as in a
    box with two ghost planes, bit for bit, and zero everywhere else."""
    from ppm_legacy_amd import core
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    torch.cuda.empty_cache()
    N, g = 8, 2
    e0 = N + 1 + 2 * g
    below = ((1 << 32) // (e0 * e0) + 40) // 2
    e2 = 2 * below + N + 1
    assert 0 < (e2 - N - 1) * e0 * e0 - (1 << 32) < 1 << 16
    mesh = core.Mesh(3, N + 1)
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand((700, 3), dtype=torch.float32, device="cuda", generator=gen) * 0.999
    if not unordered:
        c = (x * N).long()
        x = x[torch.argsort(c[:, 0] + N * (c[:, 1] + N * c[:, 2]))].contiguous()
    u = torch.randn((700, 1), dtype=torch.float32, device="cuda", generator=gen)
    small = torch.full((e0, e0, e0, 1), 7.0, dtype=torch.float32, device="cuda")
    core.p2m(mesh, x, u, small, [-g] * 3, prec=core.PREC_F32)
    big = torch.full((e2, e0, e0, 1), 7.0, dtype=torch.float32, device="cuda")
    try:
        core.p2m(mesh, x, u, big, [-g, -g, -below], prec=core.PREC_F32)
        assert torch.equal(big[below - g:below - g + e0], small)
        big[below - g:below - g + e0] = 0
        assert not any(bool((part != 0).any()) for part in big.split(1 << 21))
    finally:
        del big
        torch.cuda.empty_cache()
