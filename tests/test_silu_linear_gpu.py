"""silu(g) u of [g | u] = x w^T on the tiles of the grouped expert product without a plan (csrc/seq/moe.hip): a part-filled last row tile, one row, feature counts
around a tile and such as whole-row stores cannot take, rows of a wider matrix, more tiles than workgroups, and the layer that takes this way."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tm", [64, 256])
@pytest.mark.parametrize("n,ff,K", [(1, 128, 64), (255, 70, 128), (257, 129, 192), (1000, 768, 1024), (5000, 3072, 128), (70, 8200, 64), (0, 128, 64)])
def test_activation_leaves_with_the_product(tm, n, ff, K):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(n + ff)
    x = torch.randn(n, K + 64, generator=g).to(torch.bfloat16).cuda()[:, :K]
    w = (torch.randn(2 * ff, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
    room = torch.full((n + 300, ff), 7.0, dtype=torch.bfloat16, device="cuda")
    assert ops_seq.silu_linear_fits(x, w) or n == 0
    ops_seq.silu_linear(x, w, tm, room[:n])
    y = x.double() @ w.double().T
    want = torch.nn.functional.silu(y[:, :ff]) * y[:, ff:]
    # one rounding of the result to bfloat16: 2^-9 at most per value
    assert n == 0 or ((room[:n].double() - want).norm() / want.norm()).item() <= 2.0 ** -8
    assert (room[n:] == 7.0).all()


def test_layer_takes_it_where_the_rule_says():
    from nano_vllm_amd import ops_seq
    from nano_vllm_amd.layers import MergedColumnParallelLinear
    torch.manual_seed(0)
    layer = MergedColumnParallelLinear(512, [1024, 1024]).to(torch.bfloat16).cuda()
    layer.weight.data.copy_(torch.randn(2048, 512) / 512 ** 0.5)
    n = 3000
    assert ops_seq.silu_linear_rows(n, 1024, 512)
    x = torch.randn(n, 512).to(torch.bfloat16).cuda()
    y = x.double() @ layer.weight.double().T
    want = torch.nn.functional.silu(y[:, :1024]) * y[:, 1024:]
    for _ in range(2):
        got = layer.forward_silu(x)
    assert ((got.double() - want).norm() / want.norm()).item() <= 2.0 ** -8
