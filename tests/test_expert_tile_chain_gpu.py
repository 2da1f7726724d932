"""The pipelined grouped expert products (csrc/seq/moe.hip) where a workgroup computes several tiles one behind the other: more tiles than workgroups,
part-filled and unused row tiles between and behind them, reductions of exactly as many steps as the ring has buffers and one more, the last feature tile
part-filled, feature counts that whole-row stores cannot take, and fewer steps than buffers (a workgroup per tile)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mode", ["glu", "rows"])
@pytest.mark.parametrize("tm,counts,nout,pieces", [
    (256, [1300, 0, 1, 600, 257], 6400, 2), (256, [1100, 900], 9000, 3), (256, [2300], 7300, 1),
    (128, [700, 129, 0, 500], 6152, 3), (128, [1000, 3], 8196, 4), (64, [300, 65, 1, 700], 8192, 2), (64, [500, 200], 12292, 3),
    (16, [100, 17, 0, 1, 150], 4096, 4), (16, [90, 33], 8200, 5)])
def test_one_workgroup_computes_tile_after_tile(dtype, mode, tm, counts, nout, pieces):
    from nano_vllm_amd import ops_seq
    K = pieces * (64 if dtype == torch.bfloat16 else 32)
    E, n = len(counts), sum(counts)
    g = torch.Generator().manual_seed(nout + pieces)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(n, generator=g)].to(torch.int32).cuda()
    x = torch.randn(n, K, generator=g).to(dtype).cuda()
    w = (torch.randn(E, (2 if mode == "glu" else 1) * nout, K, generator=g) / K ** 0.5).to(dtype).cuda()
    plan = ops_seq.moe_plan(ids.view(n, 1), E, tm)
    rows = plan.pair_row.view(-1).long()
    src = x
    if mode == "rows":
        src = torch.full((plan.cap, K), float("nan"), dtype=dtype, device="cuda")
        src[rows] = x
    out = torch.full((plan.cap, nout), 7.0, dtype=dtype, device="cuda")
    for _ in range(2):
        ops_seq.moe_gemm(src, w, plan, mode == "glu", out)
    worst = 0.0
    for e in range(E):
        mine = (ids == e).nonzero().view(-1)
        y = x[mine].double() @ w[e].double().T
        want = torch.nn.functional.silu(y[:, :nout]) * y[:, nout:] if mode == "glu" else y
        worst = max(worst, ((out[rows[mine]].double() - want).norm() / want.norm()).item()) if len(mine) else worst
    # bfloat16: one rounding of the result (2^-9 at most per value); 32-bit: sums of up to 320 products, each step 2^-24
    assert worst <= (2.0 ** -8 if dtype == torch.bfloat16 else 2e-6), worst
    untouched = torch.ones(plan.cap, dtype=torch.bool, device="cuda")
    untouched[rows] = False
    assert (out[untouched] == 7.0).all()                                # padding rows are not written
