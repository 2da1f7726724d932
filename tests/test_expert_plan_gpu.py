"""The plan of the expert products, by one workgroup and by many: step sizes around the rule between them and around a workgroup's share,
from one expert to as many as there can be, pass-through choices, experts without rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,tm", [(1, 16), (4, 64), (16, 16), (17, 128), (30, 256), (64, 64), (65, 128), (1024, 16)])
@pytest.mark.parametrize("n,top", [(1, 1), (6143, 1), (6144, 1), (2049, 3), (4096, 2), (13550, 4)])
def test_every_pair_has_a_row_of_its_expert(n, top, experts, tm):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(n + experts)
    ids = torch.randint(0, experts + 2, (n, top), generator=g).to(torch.int32)          # the last two: pass-through choices
    ids[ids == experts // 2] = experts                                                  # and an expert nobody chose
    plan = ops_seq.moe_plan(ids.cuda(), experts, tm)
    flat, rows = ids.view(-1).long(), plan.pair_row.cpu().view(-1).long()
    kept = flat < experts
    assert (rows[~kept] == -1).all() and rows[kept].unique().numel() == int(kept.sum())
    token, tile = plan.row_token.cpu(), plan.tile_expert.cpu()
    assert torch.equal(token[rows[kept]].long(), (torch.arange(n * top) // top)[kept])
    assert torch.equal(tile[rows[kept] // tm].long(), flat[kept])
    assert int((token >= 0).sum()) == int(kept.sum())
    counts = torch.bincount(flat[kept], minlength=experts)
    assert torch.equal(torch.bincount(tile[tile >= 0].long(), minlength=experts), (counts + tm - 1) // tm)
