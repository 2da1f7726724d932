"""Means over blocks of positions (csrc/seq/attn_pool.hip) in steps whose columns are shared by eight, by some and by one workgroup: more columns than the shares take at
once, no whole turn of them, blocks that cross pages, tokens without a place."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,G,d,dv,block,pool", [(50, 8, 128, 128, 32, 16), (700, 3, 40, 24, 16, 12), (2600, 2, 128, 64, 64, 16), (9000, 1, 72, 136, 16, 5)])
def test_means_of_blocks(n, G, d, dv, block, pool, dtype):
    from nano_vllm_amd import ops_seq
    from nano_vllm_amd.ops_seq import Portions
    g = torch.Generator().manual_seed(n)
    pages = -(-n // block)
    bt = torch.randperm(pages, generator=g).to(torch.int32).view(1, -1).cuda()
    kc, vc = torch.randn(pages * block, G, d, generator=g).to(dtype).cuda(), torch.randn(pages * block, G, dv, generator=g).to(dtype).cuda()
    pos = torch.arange(n, device="cuda")
    slots = (bt[0, pos // block].long() * block + pos % block).to(torch.int32)
    off = 3 * pool - 1                                                  # the end of block 2 is no token of this step's cache
    slots[off] = -1
    i = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    por = Portions(i([0, n]), i([0]), i([0]), torch.zeros(n, dtype=torch.int32, device="cuda"), 1, n, n)
    rows = ops_seq.pool_rows(block, pool) * pages
    pk, pv = torch.full((rows, G * d), 9.0, device="cuda", dtype=dtype), torch.full((rows // 8, G * dv, 8), 9.0, device="cuda", dtype=dtype)
    ops_seq.pool_blocks(kc, vc, G, d, dv, block, pool, slots, pos, bt, por, pk, pv)
    K = kc[(bt[0, pos // block].long() * block + pos % block)].double().view(n, -1)
    V = vc.view(pages, G * dv, block)[bt[0, pos // block].long(), :, pos % block].double()          # (transposed inside a page)
    for b in range(n // pool):
        page = (8 * (b // 8) * pool + pool - 1) // block                # a unit of eight blocks lies with the page its first block ends in
        first = 0 if page * block < pool else (page * block - pool + 8 * pool) // (8 * pool)
        unit = int(bt[0, page]) * (ops_seq.pool_rows(block, pool) // 8) + b // 8 - first
        span = slice(b * pool, (b + 1) * pool)
        for got, src in ((pk[unit * 8 + b % 8], K[span]), (pv[unit, :, b % 8], V[span])):
            if b == 2:
                assert (got == 9.0).all()
                continue
            # a sum of `pool` numbers, a product and one rounding to the type
            tol = (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23) * src.mean(0).abs() + (pool + 1) * 2.0 ** -24 * src.abs().mean(0)
            assert ((got.double() - src.mean(0)).abs() <= tol).all(), b
