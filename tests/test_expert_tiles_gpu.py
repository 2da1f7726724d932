"""The pipelined grouped expert products (csrc/seq/moe.hip) at the edges of their tiles: every tile height, feature counts around a tile and
not a multiple of a store, reductions from one step of 128 bytes to more steps than the ring has buffers, experts with no row, one row,
exactly a tile and one row more, and input rows that are part of wider ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mode", ["glu", "relu2", "rows"])
@pytest.mark.parametrize("tm,nout,pieces", [(16, 16, 1), (16, 129, 5), (16, 70, 4), (64, 128, 2), (64, 333, 3), (128, 256, 3), (128, 70, 7),
                                            (256, 127, 2), (256, 514, 1), (256, 256, 3)])
def test_grouped_products_at_tile_edges(dtype, mode, tm, nout, pieces):
    from nano_vllm_amd import ops_seq
    K = pieces * (64 if dtype == torch.bfloat16 else 32)
    counts = [0, 1, tm, tm + 1, 5]                                      # rows per expert
    E, n = len(counts), sum(counts)
    g = torch.Generator().manual_seed(nout * 7 + pieces)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(n, generator=g)].to(torch.int32)
    wide = torch.randn(n, K + 64, generator=g).to(dtype).cuda()
    x = wide[:, :K]                                                     # rows of a wider matrix
    w = (torch.randn(E, (2 if mode == "glu" else 1) * nout, K, generator=g) / K ** 0.5).to(dtype).cuda()
    plan = ops_seq.moe_plan(ids.view(n, 1).cuda(), E, tm)
    rows = plan.pair_row.view(-1).long()
    if mode == "rows":                                                  # the input holds the planned rows; padding rows hold NaN
        src = torch.full((plan.cap, K), float("nan"), dtype=dtype, device="cuda")
        src[rows] = x
    else:
        src = x
    out = torch.full((plan.cap, nout), 7.0, dtype=dtype, device="cuda")
    ops_seq.moe_gemm(src, w, plan, mode == "glu", out, relu2=mode == "relu2")
    y = torch.einsum("nk,nfk->nf", x.double(), w.double()[ids.long().cuda()])
    want = torch.nn.functional.silu(y[:, :nout]) * y[:, nout:] if mode == "glu" else y.clamp(min=0) ** 2 if mode == "relu2" else y
    err = ((out[rows].double() - want).norm() / want.norm()).item()
    # bfloat16: one rounding of the result (2^-9 at most per value); 32-bit: sums of up to 448 products, each step 2^-24
    assert err <= (2.0 ** -8 if dtype == torch.bfloat16 else 2e-6), err
    untouched = torch.ones(plan.cap, dtype=torch.bool, device="cuda")
    untouched[rows] = False
    assert (out[untouched] == 7.0).all()                                # padding rows are not written
