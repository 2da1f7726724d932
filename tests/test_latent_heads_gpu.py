"""Latent attention's products per head (csrc/seq/latent_heads.hip): every size of the reduction and of the result, rows that are no multiple of a wavefront's 32 or a
workgroup's 128, one row and none, more rows than one pass of a workgroup, and the part behind, turned in pairs or in halves, wholly, partly or not at all."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [64, 128, 192, 256])
@pytest.mark.parametrize("N", [64, 128, 192, 256])
@pytest.mark.parametrize("turned", [True, False])
def test_products_per_head(K, N, turned):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(K + N)
    for n, H in ((0, 2), (1, 1), (33, 5), (129, 3), (3000, 130)):
        x = torch.randn(n, H, K, generator=g).to(torch.bfloat16).cuda()
        w = (torch.randn(H, *((K, N) if turned else (N, K)), generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
        room = torch.full((n + 40, H, N + 8), 5.0, dtype=torch.bfloat16, device="cuda")
        ops_seq.latent_heads(x, w, room[:n, :, :N], turned)
        wf = (w if turned else w.transpose(1, 2)).contiguous().double()
        want = torch.matmul(x.double().transpose(0, 1).contiguous(), wf).transpose(0, 1)
        # one rounding of the result to bfloat16: 2^-9 of it, in the norm
        assert n == 0 or ((room[:n, :, :N].double() - want).norm() / want.norm()).item() <= 2.0 ** -8, (n, H)
        assert (room[n:] == 5.0).all() and (room[:, :, N:] == 5.0).all()


@pytest.mark.parametrize("dr,dims,halves", [(64, 64, False), (64, 64, True), (64, 20, True), (24, 8, False), (40, 0, False)])
def test_part_behind_turns_as_rotate_heads_does(dr, dims, halves):
    from nano_vllm_amd import ops_seq
    n, H, K, N, qr = 300, 3, 128, 192, 96
    g = torch.Generator().manual_seed(dr + dims)
    x = torch.randn(n, H, K + dr, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(H, K, N, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
    pos = torch.randint(0, 5000, (n,), generator=g).cuda()
    rot = ops_seq.Rotation((10000.0 ** -torch.linspace(0, 1, dims // 2)).cuda(), halves, 1.25) if dims else None
    turn = torch.empty(n, dims // 2, 2, dtype=torch.float32, device="cuda") if dims else None
    if dims:                                                            # a layer without cache entries of its own still gives the angles
        proj = torch.randn(n, qr, generator=g).to(torch.bfloat16).cuda()
        ops_seq.latent_prep(proj, 0, qr, torch.ones(qr, dtype=torch.bfloat16, device="cuda"), torch.empty_like(proj), 1e-6, -1, 0, dr, None, pos, rot, turn=turn)
    y = torch.zeros(n, H, N + dr, dtype=torch.bfloat16, device="cuda")
    ops_seq.latent_heads(x, w, y, True, dr, rot, turn)
    want = torch.zeros(n, H, dr, dtype=torch.bfloat16, device="cuda")
    ops_seq.rotate_heads(x[:, :, K:], want, pos, rot)
    assert torch.equal(y[:, :, N:], want)
