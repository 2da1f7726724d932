"""Latent attention of prompts with the products per head in the attention kernel (nvs_latent_prompt) against the calls it stands for, latent_heads, the scalar
attention kernel and, with W_uv, latent_heads again: portions around the tiles of 32 queries and 64 keys, every number of heads a workgroup takes, windows, gates, part of the rotation or none, and pages
whose unused places hold infinities and NaN; then which steps take it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def inputs(H, lens, ctx, dims, gate, page, seed, room=0, halves=False):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g)
    n, total = sum(lens), [a + b for a, b in zip(lens, ctx)]
    need = [-(-t // page) for t in total]
    ids = torch.randperm(sum(need) + 2, generator=g)[:sum(need)].split(need)
    table = torch.full((len(lens), max(need) + 1), -1, dtype=torch.int32)
    pages = sum(need) + 2
    k, v = rand(pages, page, 1, 256), rand(pages, 1, 192, page)
    for row, (mine, t) in enumerate(zip(ids, total)):
        table[row, :len(mine)] = mine.to(torch.int32)
        if t % page:                                        # what an earlier request left behind the end
            k[mine[-1], t % page:] = float("nan")
            v[mine[-1], :, :, t % page:] = float("inf")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    por = ops_seq.Portions(i32([0] + lens).cumsum(0).to(torch.int32), i32(ctx), i32(list(range(len(lens)))),
                           torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens)).to(torch.int32).cuda(), len(lens), n, max(lens))
    bf = lambda x: x.to(BF).cuda()
    q = bf(rand(n, H * 192 + room))[:, :H * 192].view(n, H, 192)
    uk = bf(rand(H, 128, 192) / 128 ** 0.5)
    rot = ops_seq.Rotation((1000.0 ** (-torch.arange(dims // 2) / max(dims // 2, 1))).float().cuda(), halves) if dims else None
    angle = torch.cat([torch.arange(c, c + m) for m, c in zip(lens, ctx)])[:, None] * (rot.freq.cpu() if dims else torch.zeros(0))
    turn = torch.stack((angle.cos(), angle.sin()), -1).float().contiguous().cuda() if dims else None
    gates = bf(rand(n, H + 8))[:, :H] if gate else None
    return por, q, uk, rot, turn, gates, bf(k).view(-1, 1, 256), bf(v).view(-1, 1, 192), table.cuda()


CASES = [
    dict(H=16, lens=[1, 31, 32, 33, 63, 64, 65, 129], ctx=[0] * 8, dims=64),
    dict(H=8, lens=[200, 40, 96], ctx=[63, 64, 1], window=33, dims=48, gate=True, room=8),
    dict(H=3, lens=[90, 70], ctx=[0, 130], dims=0, gate=True),
    dict(H=4, lens=[300], ctx=[5], window=64, dims=16, page=256),
    dict(H=2, lens=[65, 64], ctx=[100, 0], dims=64, gate=True, window=1000),
    dict(H=32, lens=[40, 700], ctx=[700, 0], window=100, dims=64, page=128),
    dict(H=1, lens=[17] * 70, ctx=list(range(70)), dims=32, halves=True),
    dict(H=16, lens=[200, 77], ctx=[0, 9], dims=64, halves=True),
    dict(H=8, lens=[70], ctx=[0], dims=48, halves=True),
    dict(H=8, lens=[35], ctx=[3], dims=16, halves=True),
    dict(H=5, lens=[2, 300], ctx=[0, 0], window=1, dims=64),
]


@pytest.mark.parametrize("values", [False, True])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_agrees_with_the_calls_it_stands_for(case, values):
    from nano_vllm_amd import ops_seq
    kw = dict(dict(gate=False, page=64, room=0, window=0, halves=False), **CASES[case])
    H, window, page = kw["H"], kw["window"], kw["page"]
    por, q, uk, rot, turn, gates, k, v, table = inputs(H, kw["lens"], kw["ctx"], kw["dims"], kw["gate"], page, case, kw["room"], kw["halves"])
    uv = (torch.randn(H, 128, 192, generator=torch.Generator().manual_seed(50 + case)) / 192 ** 0.5).to(BF).cuda()
    room = torch.full((por.n + 40, H * (128 if values else 192)), 9.0, dtype=BF, device="cuda")
    got = room[:por.n]
    ops_seq.latent_prompt(q, uk, uv if values else None, rot, turn, gates, k, v, table, page, por, 192 ** -0.5, window, got)
    assert (room[por.n:] == 9.0).all()
    qf, want = torch.empty(por.n, H, 256, dtype=BF, device="cuda"), torch.empty(por.n, H * 192, dtype=BF, device="cuda")
    ops_seq.latent_heads(q, uk, qf, True, 64, rot, turn)
    lib = ops_seq.load_library()
    lib.nvs_window_attn_force_scalar(1)
    try:
        ops_seq.window_attn(qf.view(por.n, -1), None, 1e-6, gates, k, v, table, page, por, H, 1, 256, 192, 192 ** -0.5, window, want, gate_per_head=True)
    finally:
        lib.nvs_window_attn_force_scalar(0)
    if values:
        lat, want = want.view(por.n, H, 192), torch.empty(por.n, H, 128, dtype=BF, device="cuda")
        ops_seq.latent_heads(lat, uv, want, False)
        want = want.view(por.n, -1)
    got, want = got.double(), want.double()
    assert torch.isfinite(want).all()
    # both round the finished query and the result to 8 bits; the matrix cores round the weights too (2^-9 each, averaged over the keys); the latent result in
    # front of W_uv is rounded on either side
    err = ((got - want).norm() / want.norm()).item()
    assert err <= 2.0 ** -7, err
    assert ((got - want).abs().max() / want.pow(2).mean().sqrt()).item() <= 0.1


@pytest.mark.parametrize("values", [False, True])
def test_no_further_from_the_exact_sum_than_the_calls_it_stands_for(values):
    """One rounding of the finished query instead of two; the same ones behind it."""
    from nano_vllm_amd import ops_seq
    H, T, page = 8, 500, 64
    mine = theirs = 0.0
    for seed in range(4):
        por, q, uk, rot, turn, _, k, v, table = inputs(H, [T], [0], 64, False, page, 100 + seed)
        got, two = torch.empty(T, H * 192, dtype=BF, device="cuda"), torch.empty(T, H * 192, dtype=BF, device="cuda")
        uv = (torch.randn(H, 128, 192, generator=torch.Generator().manual_seed(seed)) / 192 ** 0.5).to(BF).cuda()
        if values:
            got = torch.empty(T, H * 128, dtype=BF, device="cuda")
        ops_seq.latent_prompt(q, uk, uv if values else None, rot, turn, None, k, v, table, page, por, 192 ** -0.5, 0, got)
        qf = torch.empty(T, H, 256, dtype=BF, device="cuda")
        ops_seq.latent_heads(q, uk, qf, True, 64, rot, turn)
        ops_seq.window_attn(qf.view(T, -1), None, 1e-6, None, k, v, table, page, por, H, 1, 256, 192, 192 ** -0.5, 0, two, gate_per_head=True)
        pages = table[0, :-(-T // page)].long().cpu()
        K = k.view(-1, page, 256)[pages].reshape(-1, 256)[:T].double().cpu()
        V = v.view(-1, 192, page)[pages].transpose(1, 2).reshape(-1, 192)[:T].double().cpu()
        x, c, s = q.double().cpu(), turn[..., 0].double().cpu()[:, None], turn[..., 1].double().cpu()[:, None]
        a, b = x[..., 128::2], x[..., 129::2]
        tail = torch.stack((a * c - b * s, b * c + a * s), -1).flatten(-2)
        lat = torch.stack([x[:, h, :128] @ uk[h].double().cpu() for h in range(H)], 1)
        score = torch.matmul(torch.cat((lat, tail), -1).transpose(0, 1).contiguous(), K.T.contiguous()) * 192 ** -0.5
        p = score.masked_fill(torch.ones(T, T).triu(1).bool(), -torch.inf).softmax(-1)
        want = torch.matmul(p, V)
        if values:
            want = torch.matmul(want, uv.double().cpu().transpose(1, 2).contiguous())
            lat, two = two.view(T, H, 192), torch.empty(T, H, 128, dtype=BF, device="cuda")
            ops_seq.latent_heads(lat, uv, two, False)
            two = two.view(T, -1)
        want = want.transpose(0, 1).reshape(T, -1)
        mine += ((got.double().cpu() - want).norm() / want.norm()).item()
        theirs += ((two.double().cpu() - want).norm() / want.norm()).item()
    assert mine <= theirs, (mine, theirs)


def test_which_steps_take_it():
    from nano_vllm_amd import ops_seq
    fits = ops_seq.load_library().nvs_latent_prompt_fits
    assert fits(2, 1, 16, 64) and fits(14000, 9, 16, 256) and fits(300, 9, 32, 64)
    assert not fits(1, 1, 16, 64) and not fits(64, 64, 16, 256)                  # single tokens
    assert not fits(300, 150, 16, 64)                                            # two tokens each: heads share query tiles
    assert not fits(500, 2, 16, 32) and not fits(500, 2, 16, 96) and not fits(500, 2, 0, 64)


def test_caches_off_16_byte_boundaries_take_the_calls_it_stands_for():
    from nano_vllm_amd import ops_seq
    from nano_vllm_amd.attn_meta import reset_context, set_context
    from nano_vllm_amd.mixers import LatentAttentionMixer
    T, page, W = 70, 64, 256
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    por = ops_seq.Portions(i32([0, T]), i32([0]), i32([0]), i32([0] * T), 1, T, T)
    torch.manual_seed(3)
    torch.set_default_dtype(BF)
    try:
        mixer = LatentAttentionMixer(W, 4, 128, 64, 128, 128, 192, 192 ** -0.5, 1e-6, page).cuda()
    finally:
        torch.set_default_dtype(torch.float32)
    for p in mixer.parameters():
        p.data.copy_(torch.ones_like(p) if p.dim() == 1 else torch.randn(p.shape, device="cuda") * p.shape[-1] ** -0.5)
    x, pos = torch.randn(T, W, device="cuda").to(BF), torch.arange(T, device="cuda")
    made = {}
    try:
        with torch.inference_mode():
            for k_off, v_off in ((0, 0), (0, 4), (4, 0)):
                mixer.k_cache, mixer.v_cache = (torch.zeros(2 * page * d + 8, dtype=BF, device="cuda")[o:o + 2 * page * d].view(2 * page, 1, d) for d, o in ((256, k_off), (192, v_off)))
                set_context(True, slot_mapping=pos.to(torch.int32), block_tables=i32([[0, 1]]), portions=por)
                made[k_off, v_off] = mixer(x, pos).double()
    finally:
        reset_context()
    want = made[0, 0]
    for got in made.values():                      # as in the first test
        assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -7
