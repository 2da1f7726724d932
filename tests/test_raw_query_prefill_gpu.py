"""Prompt attention on queries as the projection leaves them (nvl_attn_prefill_varlen_raw) against the same kernel on queries finished by the q/k-norm launch:
ragged lengths around its tiles, packed and paged keys, positions that do not start at 0, with and without the norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv", [(16, 8), (8, 1), (40, 8), (4, 4)])
@pytest.mark.parametrize("lens,cached", [([1], 0), ([127, 128, 129, 31, 33, 1], 0), ([700, 5, 1024], 0), ([40, 300, 64], 256), ([3] * 70, 0), ([2047], 512)])
@pytest.mark.parametrize("norm", [False, True])
def test_agrees_with_finished_queries(hq, hkv, lens, cached, norm):
    from nano_vllm_amd import ops
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + hq)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    n, bs, top = sum(lens), 256, 4096
    qkv = rand(n, (hq + 2 * hkv) * 128 + 64)[:, :(hq + 2 * hkv) * 128]
    qw, kw = ((1 + 0.1 * torch.randn(128, generator=g, device="cuda")).bfloat16() for _ in range(2)) if norm else (None, None)
    freq = 1e6 ** (-torch.arange(0, 128, 2, device="cuda").float() / 128)
    angle = torch.arange(top, device="cuda").float()[:, None] * freq
    table = torch.cat([angle.cos(), angle.sin()], 1).contiguous()
    pos = torch.cat([torch.arange(cached, cached + m) for m in lens]).cuda()
    need = [-(-(cached + m) // bs) for m in lens]
    bt = torch.arange(sum(need), dtype=torch.int32)
    rows = [r for r in bt.split(need)]
    bt = torch.stack([torch.cat([r, r.new_full((max(need) - len(r),), -1)]) for r in rows])
    slots = torch.cat([r[torch.arange(cached, cached + m) // bs] * bs + torch.arange(cached, cached + m) % bs for r, m in zip(rows, lens)]).to(torch.int32).cuda()
    i32 = lambda x: torch.tensor([0] + x).cumsum(0).to(torch.int32).cuda()
    cu_q, cu_k, bt = i32(lens), i32([m + cached for m in lens]), bt.cuda()
    cache = rand(sum(need), hkv, bs, 128), rand(sum(need), hkv, bs, 128)

    def store(q):
        kc, vc = cache[0].clone(), cache[1].clone()
        k = torch.empty(n, hkv, 128, device="cuda", dtype=torch.bfloat16)
        ops.qknorm_rope_kvstore(qkv, pos, qw, kw, 1e-6, table, slots, q, k, kc, vc, hq, hkv)
        return k, kc, vc
    q = torch.empty(n, hq, 128, device="cuda", dtype=torch.bfloat16)
    k, kc, vc = store(q)
    k2, kc2, vc2 = store(None)
    assert torch.equal(k, k2) and torch.equal(kc, kc2) and torch.equal(vc, vc2)
    v = qkv[:, (hq + hkv) * 128:].view(n, hkv, 128)
    for paged in ([True] if cached else [False, True]):
        args = (kc, vc) if paged else (k, v)
        tables = bt if paged else None
        want = ops.attn_prefill_varlen(q, *args, cu_q, cu_k, max(lens), 128 ** -0.5, block_tables=tables)
        got = ops.attn_prefill_raw(qkv, hq, pos, qw, 1e-6, table, *args, cu_q, cu_k, max(lens), 128 ** -0.5, block_tables=tables)
        if not norm and max(lens) < 2048 and n > 0:
            assert torch.equal(got, want)                       # the same roundings throughout
        # the norm's sum is taken in another order: an entry may round to its neighbour (2^-8 of it, and few do)
        assert float((got.double() - want.double()).norm() / want.double().norm()) <= 2.0 ** -9


@pytest.mark.parametrize("hq,hkv", [(16, 8), (12, 2), (6, 2)])
@pytest.mark.parametrize("where", ["context", "shifted", "one other", "beyond the table"])
def test_positions_as_they_are_given(hq, hkv, where):
    """The table's rows are asked for at a query's place in its context before its position is known: every other position counts all the same. Lengths around the rows of a wave (16) and of a
    workgroup (64) that takes two heads, and an odd group, whose workgroups take one."""
    from nano_vllm_amd import ops
    lens, top = [15, 16, 17, 63, 64, 65, 129, 1], 300
    g = torch.Generator(device="cuda").manual_seed(hq)
    n = sum(lens)
    qkv = torch.randn(n, (hq + 2 * hkv) * 128, generator=g, device="cuda").bfloat16()
    freq = 1e6 ** (-torch.arange(0, 128, 2, device="cuda").float() / 128)
    angle = torch.arange(top, device="cuda").float()[:, None] * freq
    table = torch.cat([angle.cos(), angle.sin()], 1).contiguous()
    pos = torch.cat([torch.arange(m) for m in lens]).cuda()
    if where == "shifted":
        pos += 100
    elif where == "one other":
        pos[40], pos[n - 1] = 7, 250
    elif where == "beyond the table":
        pos[::3], pos[1::3] = -5, 2 ** 40
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    q, k = (torch.empty(n, h, 128, device="cuda", dtype=torch.bfloat16) for h in (hq, hkv))
    ops.qknorm_rope_kvstore(qkv, pos, None, None, 1e-6, table, None, q, k, None, None, hq, hkv)
    v = qkv[:, (hq + hkv) * 128:].view(n, hkv, 128)
    want = ops.attn_prefill_varlen(q, k, v, cu, cu, max(lens), 128 ** -0.5)
    got = ops.attn_prefill_raw(qkv, hq, pos, None, 1e-6, table, k, v, cu, cu, max(lens), 128 ** -0.5)
    assert torch.equal(got, want)                               # the same roundings throughout


@pytest.mark.parametrize("lens", [[64, 10, 33], [64, 65, 10], [65, 64, 64], [20] * 16, [20] * 17, [64]])
def test_short_portions_behind_pages(lens):
    """One head a workgroup up to a mean of 64 rows and 256 pairs (portion, head), two beyond: either is the call on finished queries."""
    from nano_vllm_amd import ops
    hq, hkv, page, before = 16, 8, 64, 130
    g = torch.Generator(device="cuda").manual_seed(len(lens))
    n, per = sum(lens), -(-(before + max(lens)) // page)
    qkv = torch.randn(n, (hq + 2 * hkv) * 128, generator=g, device="cuda").bfloat16()
    angle = torch.arange(512, device="cuda").float()[:, None] * 1e6 ** (-torch.arange(0, 128, 2, device="cuda").float() / 128)
    table = torch.cat([angle.cos(), angle.sin()], 1).contiguous()
    pos = torch.cat([torch.arange(before, before + m) for m in lens]).cuda()
    kc, vc = (torch.randn(per * len(lens), hkv, page, 128, generator=g, device="cuda").bfloat16() for _ in range(2))
    bt = torch.arange(per * len(lens), dtype=torch.int32, device="cuda").view(len(lens), per)
    cu_q = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    cu_k = torch.tensor([0] + [m + before for m in lens]).cumsum(0).to(torch.int32).cuda()
    q, k = (torch.empty(n, h, 128, device="cuda", dtype=torch.bfloat16) for h in (hq, hkv))
    ops.qknorm_rope_kvstore(qkv, pos, None, None, 1e-6, table, None, q, k, None, None, hq, hkv)
    want = ops.attn_prefill_varlen(q, kc, vc, cu_q, cu_k, max(lens), 128 ** -0.5, block_tables=bt)
    got = ops.attn_prefill_raw(qkv, hq, pos, None, 1e-6, table, kc, vc, cu_q, cu_k, max(lens), 128 ** -0.5, block_tables=bt)
    assert torch.equal(got, want)                               # the same roundings throughout
