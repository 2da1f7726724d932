"""Decode attention whose parts the output projection merges (nvl_paged_attn_decode_open, nvl_linear_decode_open) against float64: contexts around a tile, a part
and the largest number of parts, empty sequences between others, pages that hold NaN behind a context's end, up to 4 rows, weights in rows and in packed tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,n_out", [(16, 8, 1024), (4, 2, 128), (16, 1, 256), (24, 8, 64)])
@pytest.mark.parametrize("lens,max_ctx", [([1, 2, 31, 32], 2048), ([0, 255, 256, 257], 4096), ([33, 0], 512), ([1023, 1024, 1025], 8192), ([2047, 2049], 4096), ([9000], 16384),
                                          ([700], 768), ([90 * k + 1 for k in range(4)], 1024), ([100] * 3 + [3000], 4096)])
def test_parts_merged_by_the_projection(hq, hkv, n_out, lens, max_ctx):
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
    qkv, w = rand(b, (hq + 2 * hkv) * 128), rand(n_out, hq * 128)
    table = torch.cat([torch.ones(max_ctx, 64), torch.zeros(max_ctx, 64)], 1).cuda()          # no rotation: the reference needs none
    ctx = torch.tensor(lens, dtype=torch.int32).cuda()
    ws = torch.full((ops.paged_attn_decode_workspace_bytes(b, hq, max_ctx),), 255, dtype=torch.uint8, device="cuda")
    scale = 128 ** -0.5
    outs = []
    for packed in (False, True):
        k, v = kc.clone(), vc.clone()
        att = ops.paged_attn_decode_open(qkv, None, None, 1e-6, table, k, v, bt.cuda(), ctx, hq, scale, max_ctx, ws)
        outs.append(ops.linear_decode_open(att, ops.pack_weight_tiles(w) if packed else w, packed=packed))
    assert torch.equal(*outs)
    got = outs[0].sum(0).double()
    for i, n in enumerate(lens):
        if n == 0:
            assert not got[i].any()
            continue
        rows = torch.arange(n)
        pages, offs = bt[i, rows // bs].long().cuda(), (rows % bs).cuda()
        K, V = k[pages, :, offs].double(), v[pages, :, offs].double()                   # [n, hkv, 128], the new token's row as the launch stored it
        assert torch.equal(K[-1].bfloat16().flatten(), qkv[i, hq * 128:(hq + hkv) * 128]) and torch.equal(V[-1].bfloat16().flatten(), qkv[i, (hq + hkv) * 128:])
        s = (qkv[i, :hq * 128].double().view(hkv, G, 1, 128) * K.permute(1, 0, 2).unsqueeze(1)).sum(3) * scale
        want = w.double() @ torch.matmul(torch.softmax(s, 2), V.permute(1, 0, 2)).view(hq * 128)
        # weights and the attention's result are rounded to 8 bits each (2^-8 of its norm); a random projection keeps that to a factor of two
        assert float((got[i] - want).norm() / want.norm()) <= 2.0 ** -7, n


@pytest.mark.parametrize("n,max_ctx", [(n, 8192) for n in (4096, 4097, 4320, 4321, 4609, 5121, 7169, 7200, 8192)] + [(4097, 16384), (7200, 16384)])
def test_new_token_weighs_once(n, max_ctx):
    """Contexts just past the largest number of parts, and past multiples of it, whose new token takes about half of the weight: counted twice, it takes two thirds."""
    from nano_vllm_amd import ops
    hq, hkv, bs = 16, 8, 256
    g = torch.Generator(device="cuda").manual_seed(n)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    pages = -(-n // bs)
    kc, vc = rand(pages, hkv, bs, 128), rand(pages, hkv, bs, 128)
    bt = torch.full((1, max_ctx // bs), -1, dtype=torch.int32)
    bt[0, :pages] = torch.arange(pages)
    u, v_new = rand(hkv, 1, 128), rand(hkv, 128)
    scale = 128 ** -0.5
    # the others' scores are normal numbers: their weights add up to about n sqrt(e)
    k_new = (u[:, 0].float() * ((torch.log(torch.tensor(n * 1.65)) / scale).cuda() / u.float().pow(2).sum(2))).bfloat16()
    qkv = torch.cat([u.expand(hkv, hq // hkv, 128).reshape(-1), k_new.reshape(-1), v_new.reshape(-1)])[None].contiguous()
    table = torch.cat([torch.ones(max_ctx, 64), torch.zeros(max_ctx, 64)], 1).cuda()
    w = torch.eye(hq * 128, device="cuda").bfloat16()                               # the projection leaves the attention's result as it is
    ws = torch.full((ops.paged_attn_decode_workspace_bytes(1, hq, max_ctx),), 255, dtype=torch.uint8, device="cuda")
    att = ops.paged_attn_decode_open(qkv, None, None, 1e-6, table, kc, vc, bt.cuda(), torch.tensor([n], dtype=torch.int32).cuda(), hq, scale, max_ctx, ws)
    got = ops.linear_decode_open(att, w).sum(0).double().view(hkv, hq // hkv, 128)
    K, V = (c.permute(0, 2, 1, 3).reshape(-1, hkv, 128)[:n].double() for c in (kc, vc))
    p = torch.softmax((u.double() * K.permute(1, 0, 2)).sum(2) * scale, 1)          # [hkv, n]
    assert 0.25 < float(p[:, -1].min()) and float(p[:, -1].max()) < 0.75
    want = torch.matmul(p.unsqueeze(1), V.permute(1, 0, 2))
    # weights and result are rounded to 8 bits each; a second count of the new token moves the result by more than a tenth
    assert float((got - want).norm() / want.norm()) <= 2.0 ** -7, n
