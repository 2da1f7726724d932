"""Decode attention of few sequences (decode_few_kernel, csrc/attn_decode.hip) against float64: contexts around its tiles of 32 tokens, its wavefronts'
turns and its parts of 1,024 tokens, with and without a plan, several launches on one plan, and pages that hold NaN behind a context's end."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv", [(16, 8), (4, 2), (5, 1), (16, 1), (24, 8)])
@pytest.mark.parametrize("lens,max_ctx", [([1, 2, 31, 32], 2048), ([33, 34, 255, 256, 257], 4096), ([1023, 1024], 8192), ([1025, 1026, 1056, 0], 4096),
                                          ([2047, 2049, 3000], 4096), ([9000], 16384), ([700], 768)])
def test_contexts_around_tiles_turns_and_parts(hq, hkv, lens, max_ctx):
    from nano_vllm_amd import ops
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + hq)
    bs, b, G = 256, len(lens), hq // hkv
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    need = [-(-n // bs) for n in lens]
    ids = torch.randperm(sum(need) + 1, generator=torch.Generator().manual_seed(1))
    bt, at = torch.full((b, max_ctx // bs), -1, dtype=torch.int32), 0
    for i, k in enumerate(need):
        bt[i, :k] = ids[at:at + k].to(torch.int32)
        at += k
    kc, vc = rand(len(ids), hkv, bs, 128), rand(len(ids), hkv, bs, 128)
    for i, n in enumerate(lens):
        if n:                                                       # the new token's place and what lies behind it
            kc[bt[i, need[i] - 1], :, (n - 1) % bs:] = float("nan")
            vc[bt[i, need[i] - 1], :, (n - 1) % bs:] = float("inf")
    qkv = rand(b, (hq + 2 * hkv) * 128)
    table = torch.cat([torch.ones(max_ctx, 64), torch.zeros(max_ctx, 64)], 1).cuda()          # no rotation: the reference needs none
    ctx = torch.tensor(lens, dtype=torch.int32).cuda()
    ws = torch.zeros(ops.paged_attn_decode_workspace_bytes(b, hq, max_ctx), dtype=torch.uint8, device="cuda")
    scale = 128 ** -0.5

    def run(plan):
        k, v, lse = kc.clone(), vc.clone(), torch.zeros(b, hq, device="cuda")
        o = ops.paged_attn_decode_fused(qkv, None, None, 1e-6, table, k, v, bt.cuda(), ctx, hq, scale, max_ctx, ws, plan=plan, lse=lse)
        return o, lse, k, v
    plan = ops.decode_plan(ctx, hq, hkv, max_ctx)
    got, lse, k, v = run(plan)
    for other in (plan, plan, None):
        o2, lse2, _, _ = run(other)
        assert torch.equal(o2, got) and torch.equal(lse2, lse)
    for i, n in enumerate(lens):
        if n == 0:
            assert not got[i].any() and bool(torch.isneginf(lse[i]).all())
            continue
        rows = torch.arange(n)
        pages, offs = bt[i, rows // bs].long().cuda(), (rows % bs).cuda()
        K, V = k[pages, :, offs].double(), v[pages, :, offs].double()                   # [n, hkv, 128], the new token's row as the launch stored it
        assert torch.equal(K[-1].bfloat16().flatten(), qkv[i, hq * 128:(hq + hkv) * 128]) and torch.equal(V[-1].bfloat16().flatten(), qkv[i, (hq + hkv) * 128:])
        s = (qkv[i, :hq * 128].double().view(hkv, G, 1, 128) * K.permute(1, 0, 2).unsqueeze(1)).sum(3) * scale
        want = torch.matmul(torch.softmax(s, 2), V.permute(1, 0, 2)).view(hq, 128)
        assert float((lse[i].double() - torch.logsumexp(s, 2).flatten()).abs().max()) <= 1e-4        # 32-bit sums of exact products
        # weights and result are rounded to 8 bits each
        assert float((got[i].double() - want).norm() / want.norm()) <= 2.0 ** -8, n


@pytest.mark.parametrize("hq,hkv", [(16, 8), (4, 2), (5, 1), (24, 8)])
@pytest.mark.parametrize("b,hi,max_ctx", [(12, 500, 1536), (12, 500, 4096), (16, 40, 1024), (8, 1500, 2048), (40, 300, 512)])
def test_pages_that_hold_no_numbers_behind_a_context(b, hi, max_ctx, hq, hkv):
    """Steps of this kernel and of the one of equal shares: what lies behind a context's end is not read into its result."""
    from nano_vllm_amd import ops
    g = torch.Generator(device="cuda").manual_seed(b + hq)
    bs, G, scale = 256, hq // hkv, 128 ** -0.5
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    lens = [1 + (hi - 1) * i // (b - 1) for i in range(b)]
    need = [-(-n // bs) for n in lens]
    bt, at = torch.full((b, max_ctx // bs), -1, dtype=torch.int32), 0
    for i, k in enumerate(need):
        bt[i, :k] = torch.arange(at, at + k)
        at += k
    kc, vc = rand(at, hkv, bs, 128), rand(at, hkv, bs, 128)
    for i, n in enumerate(lens):
        kc[bt[i, need[i] - 1], :, (n - 1) % bs:] = float("nan")
        vc[bt[i, need[i] - 1], :, (n - 1) % bs:] = float("inf")
    qkv, ctx = rand(b, (hq + 2 * hkv) * 128), torch.tensor(lens, dtype=torch.int32).cuda()
    table = torch.cat([torch.ones(max_ctx, 64), torch.zeros(max_ctx, 64)], 1).cuda()
    ws = torch.full((ops.paged_attn_decode_workspace_bytes(b, hq, max_ctx),), 255, dtype=torch.uint8, device="cuda")
    plan = ops.decode_plan(ctx, hq, hkv, max_ctx)
    before = plan.clone()
    for p in (plan, None):
        k, v = kc.clone(), vc.clone()
        got = ops.paged_attn_decode_fused(qkv, None, None, 1e-6, table, k, v, bt.cuda(), ctx, hq, scale, max_ctx, ws, plan=p)
        for i, n in enumerate(lens):
            rows = torch.arange(n)
            pages, offs = bt[i, rows // bs].long().cuda(), (rows % bs).cuda()
            K, V = k[pages, :, offs].double(), v[pages, :, offs].double()
            s = (qkv[i, :hq * 128].double().view(hkv, G, 1, 128) * K.permute(1, 0, 2).unsqueeze(1)).sum(3) * scale
            want = torch.matmul(torch.softmax(s, 2), V.permute(1, 0, 2)).view(hq, 128)
            assert float((got[i].double() - want).norm() / want.norm()) <= 2.0 ** -8, (i, n)          # weights and result are rounded to 8 bits each
    assert torch.equal(plan, before)                                # launches of several streams may share a plan: none writes it
