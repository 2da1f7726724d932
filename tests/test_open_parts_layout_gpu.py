"""The parts that a decode step's attention leaves open lie where include/nvl.h says, and the output projection merges parts laid out by that text alone: both entries, in
parts of eight tiles and in fours, for the contexts at which the two rules differ."""
import functools

import pytest
import torch

pytestmark = pytest.mark.gpu
LENS = [[257, 700, 0, 30], [1200], [513, 2000, 1025], [3000, 260]]


def header_parts(tokens, parts, fours):
    """(number of parts, tiles of each) of a context, from the text in include/nvl.h."""
    t = -(-tokens // 32)
    n = -(-t // 8)
    if n <= 1:
        return 1, t
    r = -(-n // 4) * 4 if fours else n
    if not (r == n <= parts):
        n = -(-t // -(-t // min(r, parts)))
    return n, -(-t // n)


@pytest.mark.parametrize("fours", [False, True])
@pytest.mark.parametrize("lens", LENS)
def test_projection_merges_parts_of_the_documented_layout(lens, fours):
    """Parts that were not left are NaN: a projection that cuts a context otherwise meets them."""
    from nano_vllm_amd import ops
    hq, n_out, b, longest = 16, 256, len(lens), 4096
    parts = ops.open_parts(b, 8, longest, fours=True) if fours else ops.open_parts(b, 8, longest)
    g = torch.Generator(device="cuda").manual_seed(sum(lens))
    po = torch.full((b, hq, parts, 128), float("nan"), device="cuda")
    ml = torch.full((b, hq, parts, 2), float("nan"), device="cuda")
    whole = torch.zeros(b, hq, 128, dtype=torch.bfloat16, device="cuda")
    x = torch.zeros(b, hq * 128, dtype=torch.float64, device="cuda")
    for i, tokens in enumerate(lens):
        n = header_parts(tokens, parts, fours)[0]
        if n == 1:
            whole[i] = torch.randn(hq, 128, generator=g, device="cuda") * (tokens > 0)
            x[i] = whole[i].double().flatten()
            continue
        po[i, :, :n] = torch.randn(hq, n, 128, generator=g, device="cuda")
        ml[i, :, :n, 0] = torch.randn(hq, n, generator=g, device="cuda")
        ml[i, :, :n, 1] = torch.rand(hq, n, generator=g, device="cuda") + 1
        weight = torch.exp2(ml[i, :, :n, 0].double())
        x[i] = ((po[i, :, :n].double() * weight[..., None]).sum(1) / (ml[i, :, :n, 1].double() * weight).sum(1)[:, None]).flatten()
    room = torch.cat([t.contiguous().view(torch.uint8).flatten() for t in (po, ml, whole)])
    att = ops.OpenAttention(room, torch.tensor(lens, dtype=torch.int32, device="cuda"), b, hq, parts, *([True] if fours else []))
    w = torch.randn(n_out, hq * 128, generator=g, device="cuda").bfloat16()
    got, want = ops.linear_decode_open(att, w).sum(0).double(), x @ w.double().T
    for i, tokens in enumerate(lens):
        if tokens == 0:
            assert not got[i].any()
        else:                             # the merged row is rounded to 8 bits (2^-9 of a value); a random projection keeps that to a factor of two
            assert float((got[i] - want[i]).norm() / want[i].norm()) <= 2.0 ** -8, tokens


@pytest.mark.parametrize("fours", [False, True])
@pytest.mark.parametrize("lens", LENS)
def test_attention_leaves_the_documented_layout(lens, fours):
    """Every part by itself: numerators, maximum and sum over its tiles' tokens."""
    from nano_vllm_amd import ops
    hq, hkv, b, longest, bs, scale = 16, 8, len(lens), 4096, 256, 128 ** -0.5
    g = torch.Generator(device="cuda").manual_seed(sum(lens))
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    pages = [-(-n // bs) for n in lens]
    kc, vc = rand(sum(pages) + 1, hkv, bs, 128), rand(sum(pages) + 1, hkv, bs, 128)
    bt = torch.zeros(b, longest // bs, dtype=torch.int32)
    for i, n in enumerate(pages):
        bt[i, :n] = torch.arange(n) + sum(pages[:i])
    qkv = rand(b, (hq + 2 * hkv) * 128)
    table = torch.cat([torch.ones(longest, 64), torch.zeros(longest, 64)], 1).cuda()          # no rotation
    ws = torch.full((ops.paged_attn_decode_workspace_bytes(b, hq, longest),), 255, dtype=torch.uint8, device="cuda")
    att = ops.paged_attn_decode_open(qkv, None, None, 1e-6, table, kc, vc, bt.cuda(), torch.tensor(lens, dtype=torch.int32).cuda(), hq, scale, longest, ws,
                                     *([True] if fours else []))
    P = att.parts
    po = ws[:b * hq * P * 512].view(torch.float32).view(b, hq, P, 128)
    ml = ws[b * hq * P * 512:b * hq * P * 520].view(torch.float32).view(b, hq, P, 2)
    for i, tokens in enumerate(lens):
        n, per = header_parts(tokens, P, fours)
        if n == 1:
            continue
        K, V = (c[bt[i, :pages[i]].long().cuda()].permute(0, 2, 1, 3).reshape(-1, hkv, 128)[:tokens].double().repeat_interleave(hq // hkv, 1) for c in (kc, vc))
        s = (K * qkv[i, :hq * 128].double().view(hq, 128)).sum(2).T * (scale * 1.4426950408889634)         # [hq, tokens], base 2
        for p in range(n):
            a, z = p * per * 32, min((p + 1) * per * 32, tokens)
            assert a < z
            weight = torch.exp2(s[:, a:z] - ml[i, :, p, :1].double())
            # sums of 32-bit weights, whose exponents (up to 2^4 here) are rounded to 2^-20; weights are rounded to 8 bits for the numerators
            assert torch.allclose(weight.sum(1), ml[i, :, p, 1].double(), rtol=1e-4), (tokens, p)
            want = torch.matmul(weight[:, None], V[a:z].permute(1, 0, 2))[:, 0]
            assert float((po[i, :, p].double() - want).norm() / want.norm()) <= 2.0 ** -7, (tokens, p)


@pytest.fixture
def in_fours(monkeypatch):
    from nano_vllm_amd import ops
    monkeypatch.setattr(ops, "paged_attn_decode_open", functools.partial(ops.paged_attn_decode_open, fours=True))


@pytest.mark.parametrize("lens,max_ctx", [([0, 255, 256, 257], 4096), ([1023, 1024, 1025], 8192), ([9000], 16384), ([700], 768), ([100] * 3 + [3000], 4096)])
def test_parts_in_fours_merged_by_the_projection(in_fours, lens, max_ctx):
    from test_open_attention_gpu import test_parts_merged_by_the_projection
    test_parts_merged_by_the_projection(16, 8, 1024, lens, max_ctx)


@pytest.mark.parametrize("n,max_ctx", [(4097, 8192), (4321, 8192), (7200, 8192), (7200, 16384)])
def test_new_token_weighs_once_in_fours(in_fours, n, max_ctx):
    from test_open_attention_gpu import test_new_token_weighs_once
    test_new_token_weighs_once(n, max_ctx)
