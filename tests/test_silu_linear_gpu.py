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


@pytest.mark.parametrize("lo,hi", [(-20.0, -10.0), (-80.0, -60.0), (-2.0, 2.0), (4.0, 30.0)])
def test_activation_keeps_the_bits_of_its_sums(lo, hi):
    """Gates of 24 bits (three 16-bit entries that add up exactly), up = 1: how many results are not the nearest bfloat16 number to silu(g). An error of k 2^-24
    crosses a rounding boundary, 2^-8 apart, k 2^-16 of the time: the limit is k = 1, two roundings of half a unit (1 + e^-g, the quotient)."""
    from nano_vllm_amd import ops_seq
    n, K = 1 << 20, 64
    g = torch.empty(n).uniform_(lo, hi, generator=torch.Generator().manual_seed(1)).cuda()
    x, left = torch.zeros(n, K, dtype=torch.bfloat16, device="cuda"), g.clone()
    for i in range(3):
        x[:, i] = (left.view(torch.int32) & -65536).view(torch.float32).bfloat16()
        left -= x[:, i].float()
    assert not left.any()
    x[:, 3] = 1.0
    w = torch.zeros(16, K, dtype=torch.bfloat16, device="cuda")
    w[:8, :3], w[8:, 3] = 1.0, 1.0
    want = torch.nn.functional.silu(g.double())
    for tm in (64, 256):
        got = ops_seq.silu_linear(x, w, tm)
        assert torch.equal(got, got[:, :1].expand_as(got))
        off = (got[:, 0].double() - want).abs() > (want.bfloat16().double() - want).abs()
        assert float(off.double().mean()) <= 2.0 ** -16, float(off.double().mean()) * 2.0 ** 16


def test_gates_beyond_the_exponential():
    from nano_vllm_amd import ops_seq
    g = torch.tensor([-3e38, -1000.0, -200.0, -90.0, -0.0, 0.0, 90.0, 200.0, 3e38, float("inf"), float("-inf")])
    x = torch.zeros(11, 64)
    x[:, 0], x[:, 1] = (g / 2).clamp(-3e38, 3e38), 1.0               # (twice the largest is an infinity)
    w = torch.zeros(16, 64)
    w[:8, 0], w[8:, 1] = 2.0, 1.0
    got = ops_seq.silu_linear(x.bfloat16().cuda(), w.bfloat16().cuda(), 64)[:, 0].float().cpu()
    assert not got[:6].any() and torch.equal(got[6:9], g[6:9].bfloat16().float()) and got[9] == float("inf") and got[10].isnan()
