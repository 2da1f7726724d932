"""The tile heights of a step's expert plan (ops_seq.moe_plan_rows): which steps take the tiles of 256 rows, which stay with moe_tile_rows, and the experts' sum
on either side of the lines against one in 64 bits, with every pair at one expert, with experts that get none and with choices that are no expert."""
import pytest
import torch

BF = torch.bfloat16


@pytest.mark.parametrize("width,ff,experts,per,want", [
    (4096, 3072, 32, 127, 128), (4096, 3072, 32, 128, 256), (1024, 768, 32, 127, 64), (1024, 768, 32, 128, 256), (2048, 512, 8, 250, 256),
    (4096, 3072, 2, 450, 128), (4096, 3072, 2, 900, 256), (8192, 1024, 4, 250, 128), (4096, 1024, 8, 180, 128), (4096, 1024, 8, 250, 256),
    (2048, 1536, 8, 180, 128), (2048, 1536, 8, 256, 256), (2048, 2048, 1, 1500, 256),
    (2048, 2048, 1, 400, 16), (1024, 768, 4, 175, 16), (96, 128, 32, 300, 128), (1024, 64, 32, 300, 64)])
def test_heights(width, ff, experts, per, want):
    from nano_vllm_amd.ops_seq import moe_plan_rows
    assert moe_plan_rows(per * experts, experts, width, ff, BF) == want


def test_calls_of_the_other_kernels_keep_their_heights():
    """32-bit rows, rows that are no whole pieces, and few rows: the tiles of 256 rows are not reached, so nothing is chosen for them."""
    from nano_vllm_amd.ops_seq import moe_plan_rows, moe_tile_rows
    for experts in (1, 4, 32, 128):
        for per in (1, 40, 127, 128, 300, 2000):
            for width, ff in ((1024, 768), (2048, 512), (4096, 3072), (1000, 520), (1024, 520), (64, 128)):
                pairs = per * experts
                assert moe_plan_rows(pairs, experts, width, ff, torch.float32) == moe_tile_rows(pairs, experts, width, ff, torch.float32)
                if per < 128 or width % 64 or ff % 64 or width < 128 or moe_tile_rows(pairs, experts, width, ff, BF) == 16:
                    assert moe_plan_rows(pairs, experts, width, ff, BF) == moe_tile_rows(pairs, experts, width, ff, BF)


@pytest.mark.gpu
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("width,ff,experts,per", [(1024, 768, 32, 127), (1024, 768, 32, 129), (2048, 1536, 8, 255), (2048, 1536, 8, 257), (4096, 192, 16, 140), (320, 640, 24, 200)])
@pytest.mark.parametrize("routing", ["even", "one", "few"])
def test_the_experts_sum(routing, width, ff, experts, per, gated):
    from nano_vllm_amd import ops_seq
    top, n = 2, per * experts // 2
    g = torch.Generator().manual_seed(width + per)
    ids = torch.randint({"even": experts, "one": 1, "few": 3}[routing], (n, top), generator=g)
    if routing == "few":
        ids = torch.where(ids == 1, experts + 1, ids + 2)                    # a choice that is no expert: the token itself
    wts = torch.rand(n, top, generator=g).cuda()
    x = torch.randn(n, width, generator=g).to(BF).cuda()
    gen = torch.Generator(device="cuda").manual_seed(ff)
    up = (torch.randn(experts, (2 if gated else 1) * ff, width, generator=gen, device="cuda") / width ** 0.5).to(BF)
    down = (torch.randn(experts, width, ff, generator=gen, device="cuda") / ff ** 0.5).to(BF)
    plan = ops_seq.moe_plan(ids.to(torch.int32).cuda(), experts, ops_seq.moe_plan_rows(n * top, experts, width, ff, BF))
    act, rows = torch.empty(plan.cap, ff, dtype=BF, device="cuda"), torch.empty(plan.cap, width, dtype=BF, device="cuda")
    ops_seq.moe_gemm(x, up, plan, gated, act, relu2=not gated)
    ops_seq.moe_gemm(act, down, plan, False, rows)
    out = torch.empty_like(x)
    ops_seq.moe_combine(rows, plan, wts, x, None, None, out)
    want = torch.zeros(n, width, dtype=torch.float64, device="cuda")
    for e in range(experts + 2):
        t, k = (ids.cuda() == e).nonzero(as_tuple=True)
        if len(t):
            y = x[t].double()
            if e < experts:
                y = y @ up[e].double().T
                y = torch.nn.functional.silu(y[:, :ff]) * y[:, ff:] if gated else y.clamp(min=0) ** 2
                y = y @ down[e].double().T
            want.index_add_(0, t, wts[t, k].double()[:, None] * y)
    err = ((out.double() - want).norm() / want.norm()).item()
    # three roundings to 8 bits one behind the other (activation, row, sum), 2^-9 each at most; the 32-bit sums are far below
    assert err <= 3 * 2.0 ** -9, err
