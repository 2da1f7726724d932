"""The attention kernel for steps of prompts (csrc/seq/attn_prompt.h) against the scalar kernel, which takes every call: portions around its tiles of
32 queries and 64 keys, behind contexts that end anywhere in a page, all masks, sinks, norms, rotations, gates and pooled blocks, and pages whose
unused places hold infinities and NaN."""
import pytest
import torch

pytestmark = pytest.mark.gpu

PAGE = 64


def call(scalar, H, G, d, dv, lens, ctx, window=0, chunk=0, rot=0, norm="", sink=False, gate=0, temp=None, pool=0, cap=0.0, seed=0):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g)
    n, total = sum(lens), [a + b for a, b in zip(lens, ctx)]
    need = [-(-t // PAGE) for t in total]
    ids = torch.randperm(sum(need) + 2, generator=g)[:sum(need)].split(need)
    table = torch.full((len(lens), max(need) + 1), -1, dtype=torch.int32)
    pages = sum(need) + 2
    k, v = rand(pages, PAGE, G, d), rand(pages, G, dv, PAGE)
    for row, (mine, t) in enumerate(zip(ids, total)):
        table[row, :len(mine)] = mine.to(torch.int32)
        if t % PAGE:                                        # what an earlier request left behind the end
            k[mine[-1], t % PAGE:] = float("nan")
            v[mine[-1], :, :, t % PAGE:] = float("inf")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    por = ops_seq.Portions(i32([0] + lens).cumsum(0).to(torch.int32), i32(ctx), i32(list(range(len(lens)))),
                           torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens)).to(torch.int32).cuda(), len(lens), n, max(lens))
    bf = lambda x: x.to(torch.bfloat16).cuda()
    q = bf(rand(n, H * d + 8))[:, :H * d]
    w = bf(1 + 0.1 * rand(H * d if norm == "rows" else d)) if norm else None
    kw = dict(gate_per_head=gate == 1, sink=rand(H).cuda() if sink else None, q_temp=temp, softcap=cap)
    if norm == "rows":
        kw["q_row"] = (0.5 + torch.rand(n, generator=g)).cuda()
    kc = bf(k).view(pages * PAGE, G, d)
    vc = bf(v).view(pages * PAGE, G, dv)
    if pool:
        rows = ops_seq.pool_rows(PAGE, pool)
        kw.update(pool=pool, pool_k=bf(rand(pages, rows, G, d)), pool_v=bf(rand(pages, rows // 8, G, dv, 8)))
    gates = bf(rand(n, H * (1 if gate == 1 else dv))) if gate else None
    freq = (1000.0 ** (-torch.arange(rot // 2) / max(rot // 2, 1))).float().cuda() if rot else None
    out = torch.full((n, H * dv), 9.0, dtype=torch.bfloat16, device="cuda")
    lib = ops_seq.load_library()
    lib.nvs_window_attn_force_scalar(1 if scalar else 0)
    try:
        ops_seq.window_attn(q, w, 1e-6, gates, kc, vc, table.cuda(), PAGE, por, H, G, d, dv, d ** -0.5, window, out, chunk, freq, **kw)
    finally:
        lib.nvs_window_attn_force_scalar(0)
    return out


CASES = [
    dict(H=4, G=2, lens=[1, 31, 32, 33, 63, 64, 65, 129], ctx=[0] * 8),
    dict(H=8, G=2, lens=[200, 40, 96], ctx=[63, 64, 1], window=33, sink=True),
    dict(H=3, G=3, lens=[90, 70], ctx=[0, 130], chunk=48, rot=128, norm="head"),
    dict(H=8, G=1, lens=[300], ctx=[5], window=64, gate=2, temp=(0.3, 16)),
    dict(H=6, G=2, lens=[65, 64], ctx=[100, 0], rot=40, gate=1, sink=True),
    dict(H=4, G=2, lens=[400, 66], ctx=[0, 333], window=40, pool=4, cap=5.0, norm="rows", sink=True),
    dict(H=4, G=4, lens=[150, 64], ctx=[700, 0], window=64, pool=16, cap=30.0, norm="rows", rot=64),
    dict(H=2, G=1, lens=[130], ctx=[0], cap=4.0),
    dict(H=1, G=1, lens=[17] * 70, ctx=[i for i in range(70)]),
]


@pytest.mark.parametrize("d,dv,case", [(128, 128, i) for i in range(len(CASES))] +
                         [(256, 192, i) for i, c in enumerate(CASES) if not (c.get("cap") or c.get("pool"))])      # (those sizes take the kernel without the extensions)
def test_prompt_kernel_agrees_with_the_scalar_kernel(d, dv, case):
    kw = dict(CASES[case], d=d, dv=dv, seed=case)
    got, want = call(False, **kw).double(), call(True, **kw).double()
    assert torch.isfinite(want).all()
    # both round the finished query and the result to 8 bits; the matrix cores round the weights too (2^-9 each, averaged over the keys)
    err = ((got - want).norm() / want.norm()).item()
    assert err <= 2.0 ** -7, err
    assert ((got - want).abs().max() / want.pow(2).mean().sqrt()).item() <= 0.1


ORDERS = [
    dict(lens=[40, 1, 0, 200, 64], ctx=[140000, 0, 0, 131050, 5], window=100),       # places beyond the first 64 x 64, a portion of nothing
    dict(lens=[(7 * i) % 90 + 1 for i in range(64)], ctx=[(37 * i) % 300 for i in range(64)]),
    dict(lens=[(7 * i) % 90 + 1 for i in range(65)], ctx=[(37 * i) % 300 for i in range(65)]),      # more than lanes: portion by portion
    dict(lens=[4100], ctx=[31], chunk=64),
]


@pytest.mark.parametrize("d,dv", [(128, 128), (256, 192)])
@pytest.mark.parametrize("case", range(len(ORDERS)))
def test_every_tile_of_every_portion_is_somebodys(d, dv, case):
    """The order of the tiles (the furthest positions first, whatever the portion) leaves none out: bounds as above."""
    kw = dict(ORDERS[case], H=2, G=1, d=d, dv=dv, seed=20 + case)
    got, want = call(False, **kw).double(), call(True, **kw).double()
    err = ((got - want).norm() / want.norm()).item()
    assert err <= 2.0 ** -7, err
    assert ((got - want).abs().max() / want.pow(2).mean().sqrt()).item() <= 0.1


def step(q, K, V, lens, ctx, H, G, d, dv, scale=1.0, window=0, sink=None, gates=None, per_head=False, page=64):
    """One call on sequences whose keys K [tokens of all, G, d] and values V [.., G, dv] lie in pages in order."""
    from nano_vllm_amd import ops_seq
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    need = [-(-(a + b) // page) for a, b in zip(lens, ctx)]
    kc = torch.zeros(sum(need), page, G, d, dtype=torch.bfloat16, device="cuda")
    vc = torch.zeros(sum(need), G, dv, page, dtype=torch.bfloat16, device="cuda")
    table = torch.zeros(len(lens), max(need), dtype=torch.int32)
    at = first = 0
    for s, (a, b) in enumerate(zip(lens, ctx)):
        T = a + b
        kc[first:first + need[s]].view(-1, G, d)[:T] = K[at:at + T].to(torch.bfloat16)
        flat = torch.zeros(need[s] * page, G, dv, dtype=torch.bfloat16, device="cuda")
        flat[:T] = V[at:at + T].to(torch.bfloat16)
        vc[first:first + need[s]] = flat.view(need[s], page, G, dv).permute(0, 2, 3, 1)
        table[s, :need[s]] = torch.arange(first, first + need[s])
        at, first = at + T, first + need[s]
    n = sum(lens)
    por = ops_seq.Portions(i32([0] + lens).cumsum(0).to(torch.int32), i32(ctx), i32(list(range(len(lens)))),
                           torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens)).to(torch.int32).cuda(), len(lens), n, max(lens))
    out = torch.full((n, H * dv), 9.0, dtype=torch.bfloat16, device="cuda")
    ops_seq.window_attn(q, None, 1e-6, gates, kc.view(-1, G, d), vc.view(-1, G, dv), table.cuda(), page, por, H, G, d, dv, scale, window, out,
                        gate_per_head=per_head, sink=sink)
    return out


SIZES = [(128, 128), (256, 192)]


@pytest.mark.parametrize("d,dv", SIZES)
@pytest.mark.parametrize("per_head", [False, True])
def test_gates_are_exact_to_their_last_bits(d, dv, per_head):
    """With one visible key the output is its value times the gate, rounded once to bfloat16: it lies between the roundings of the exact
    product less and plus six roundings of 2^-24 (a sigmoid and a product in 32 bits: its exponential takes two, sum, reciprocal and product one)."""
    g = torch.Generator(device="cuda").manual_seed(d)
    H, n = 4, 600
    v = torch.randn(n, 1, dv, generator=g, device="cuda").bfloat16()
    gates = (torch.rand(n, H * (1 if per_head else dv), generator=g, device="cuda") * 100 - 80).bfloat16()
    q = torch.randn(n, H * d, generator=g, device="cuda").bfloat16()
    got = step(q, torch.zeros(n, 1, d, device="cuda"), v, [1] * n, [0] * n, H, 1, d, dv, gates=gates, per_head=per_head).view(n, H, dv)
    want = v.double() * torch.sigmoid(gates.double().view(n, H, -1))
    lo, hi = ((want * (1 + f * 6 * 2.0 ** -24)).float().bfloat16() for f in (-1, 1))
    assert ((got >= torch.minimum(lo, hi)) & (got <= torch.maximum(lo, hi))).all()


@pytest.mark.parametrize("d,dv", SIZES)
@pytest.mark.parametrize("value", [float("-inf"), torch.finfo(torch.float32).min, -2.5e38, -1e31])
@pytest.mark.parametrize("window", [0, 33, 64, 100])
def test_a_sink_without_weight(d, dv, value, window):
    """A sink that weighs nothing changes nothing, also where a query sees no key of its workgroup's first rounds."""
    g = torch.Generator(device="cuda").manual_seed(window)
    H, lens, ctx = 2, [300, 5, 1], [0, 130, 200]
    n, total = sum(lens), sum(lens) + sum(ctx)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    args = rand(n, H * d).bfloat16(), rand(total, 1, d), rand(total, 1, dv), lens, ctx, H, 1, d, dv, d ** -0.5, window
    plain, with_sink = step(*args), step(*args, sink=torch.full((H,), value, device="cuda"))
    assert torch.isfinite(plain).all() and torch.equal(plain, with_sink)


@pytest.mark.parametrize("d,dv", SIZES)
@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("a,b,unit", [(3, 4, 1), (9, 9, 1), (-10, 10, 1), (12, 12, 2), (17, 17, 2048)])
def test_weights_of_rounds_with_different_maxima(d, dv, a, b, unit, sink):
    """Scores of 2^(|a| + b) (negative with a) plus small whole numbers, all exact: the largest moves from round to round, and the weights must
    stay on one scale however far from 0 they all lie. Weights and output are rounded to 8 bits (2^-9 each, and what they add up to)."""
    g = torch.Generator(device="cuda").manual_seed(b)
    H, T, n = 2, 500, 40
    delta = torch.randint(0, 3, (T,), generator=g, device="cuda") + torch.arange(T, device="cuda") // 64 % 5
    q, K = torch.zeros(n, H, d, device="cuda"), torch.zeros(T, 1, d, device="cuda")
    q[..., 0], q[..., 1], K[:, 0, 0], K[:, 0, 1] = 2.0 ** abs(a) * (-1 if a < 0 else 1), unit, 2.0 ** b, delta.float()
    V = torch.randn(T, 1, dv, generator=g, device="cuda").bfloat16()
    start = 2.0 ** (abs(a) + b) * (-1 if a < 0 else 1)
    s = torch.full((H,), start + 4 * unit, device="cuda") if sink else None
    got = step(q.view(n, -1).bfloat16(), K, V, [n], [T - n], H, 1, d, dv, sink=s).view(n, H, dv).double()
    score = (start + unit * delta.double()).expand(n, T).clone()
    score[torch.arange(T, device="cuda") > torch.arange(T - n, T, device="cuda")[:, None]] = -torch.inf
    extra = torch.full((n, 1), start + 4 * unit if sink else -torch.inf, dtype=torch.float64, device="cuda")
    p = torch.cat([score, extra], 1).softmax(1)[:, :-1]
    want = (p @ V[:, 0].double())[:, None].expand(n, H, dv)
    assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -7


@pytest.mark.parametrize("d,dv,H,G,pool", [(64, 64, 4, 2, 0), (64, 64, 16, 1, 0), (128, 64, 8, 1, 0), (64, 128, 2, 1, 4)])
def test_single_tokens_of_other_sizes_do_not_see_what_a_page_held_before(d, dv, H, G, pool):
    kw = dict(H=H, G=G, d=d, dv=dv, lens=[1] * 9, ctx=[0, 6, 7, 8, 62, 63, 64, 70, 199], window=40 if pool else 0, pool=pool, seed=d)
    got, want = call(False, **kw).double(), call(True, **kw).double()
    assert torch.isfinite(want).all()
    assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -7
    assert ((got - want).abs().max() / want.pow(2).mean().sqrt()).item() <= 0.1


@pytest.mark.parametrize("d,dv,H,G,nseq,cap", [(128, 128, 64, 1, 32, 0.0), (128, 128, 64, 1, 33, 0.0), (128, 128, 18, 2, 28, 0.0), (128, 128, 18, 2, 29, 0.0),
                                               (128, 128, 16, 2, 64, 5.0), (128, 128, 16, 2, 65, 5.0), (256, 192, 72, 1, 28, 0.0), (256, 192, 72, 1, 29, 0.0)])
def test_single_tokens_with_many_heads_over_a_kv_head(d, dv, H, G, nseq, cap):
    """On either side of the step where the kernel's workgroups no longer run at once and heads are packed into query tiles instead."""
    kw = dict(H=H, G=G, d=d, dv=dv, lens=[1] * nseq, ctx=[(37 * i) % 200 for i in range(nseq)], sink=True, cap=cap, seed=nseq)
    got, want = call(False, **kw).double(), call(True, **kw).double()
    assert torch.isfinite(want).all()
    assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -7
    assert ((got - want).abs().max() / want.pow(2).mean().sqrt()).item() <= 0.1


@pytest.mark.parametrize("d,dv", SIZES)
@pytest.mark.parametrize("H,G", [(3, 3), (2, 1), (4, 1), (8, 1)])
@pytest.mark.parametrize("window", [0, 40])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_a_value_that_is_not_finite_stays_with_the_tokens_around_it(d, dv, H, G, window, value):
    """A value of token j lies in a tile of 64 keys, and 32 queries go together: the products of a tile that none of them sees are left out, so
    what token j brings stays with the queries around it."""
    g = torch.Generator(device="cuda").manual_seed(H + window)
    lens, ctx = [500, 130, 31], [0, 70, 300]
    n, total = sum(lens), sum(lens) + sum(ctx)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    q, K, V = rand(n, H * d).bfloat16(), rand(total, G, d), rand(total, G, dv)
    run = lambda v: step(q, K, v, lens, ctx, H, G, d, dv, d ** -0.5, window).view(n, H, dv)
    clean = run(V)
    assert torch.isfinite(clean).all()
    for s, j in ((0, 0), (0, 70), (0, 130), (0, 319), (0, 499), (1, 5), (1, 110), (1, 199), (2, 20), (2, 330)):
        at, row = sum(lens[:s]) + sum(ctx[:s]), sum(lens[:s])
        bad = V.clone()
        bad[at + j, G - 1, dv // 2] = value
        got = run(bad)
        pos = torch.arange(ctx[s], ctx[s] + lens[s], device="cuda")
        sees = (pos >= j) & (pos - j < window if window else True)
        first = ctx[s] + torch.arange(lens[s], device="cuda") // 32 * 32
        touched = (first + 31 >= j // 64 * 64) & (first - window + 1 <= j // 64 * 64 + 63 if window else True)
        same = torch.ones(n, dtype=torch.bool, device="cuda")
        same[row:row + lens[s]] = ~touched
        assert torch.equal(got[same], clean[same]), (s, j)
        assert not torch.isfinite(got[row:row + lens[s]][sees][:, -1, dv // 2]).any(), (s, j)


@pytest.mark.parametrize("page", [64, 128, 256])
@pytest.mark.parametrize("d,dv", SIZES)
@pytest.mark.parametrize("H,G,window,sink,gated", [(4, 2, 0, False, False), (8, 1, 70, True, True), (3, 3, 0, True, False), (12, 2, 40, False, True)])
def test_prompt_kernel_against_float64(d, dv, H, G, window, sink, gated, page):
    """Rounded to 8 bits: the scaled query, the weights (2^-9 each, which average out over the keys) and the result."""
    g = torch.Generator(device="cuda").manual_seed(page + H)
    lens, ctx = [200, 33, 1, 64], [0, 300, 129, 64]
    n, total = sum(lens), sum(lens) + sum(ctx)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    q, K, V = rand(n, H * d).bfloat16(), rand(total, G, d).bfloat16(), rand(total, G, dv).bfloat16()
    s0, gates = rand(H) if sink else None, rand(n, H * dv).bfloat16() if gated else None
    got = step(q, K, V, lens, ctx, H, G, d, dv, d ** -0.5, window, sink=s0, gates=gates, page=page).view(n, H, dv).double()
    want, row, at = torch.empty_like(got), 0, 0
    for a, c in zip(lens, ctx):
        k, v = (t[at:at + a + c].double().repeat_interleave(H // G, 1).transpose(0, 1) for t in (K, V))
        score = q[row:row + a].double().view(a, H, d).transpose(0, 1) @ k.transpose(1, 2).contiguous() * d ** -0.5
        i, j = torch.arange(c, c + a, device="cuda")[:, None], torch.arange(a + c, device="cuda")
        score = score.masked_fill((j > i) | (i - j >= window if window else False), -torch.inf)
        if sink:
            score = torch.cat([score, s0.double()[:, None, None].expand(H, a, 1)], 2)
        want[row:row + a] = (score.softmax(2)[..., :a + c] @ v).transpose(0, 1)
        row, at = row + a, at + a + c
    if gated:
        want *= torch.sigmoid(gates.double()).view(n, H, dv)
    assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -7
    assert ((got - want).abs().max() / want.pow(2).mean().sqrt()).item() <= 0.1


def test_equal_pairs_turn_to_equal_bits():
    """All pairs of a query's row alike and of one frequency: their rotations are the same two 16-bit numbers whichever pair it is. Key j of the 128 in the pages shows entry j alone,
    value j counts in column j alone, so that column is the weight of the entry's score, times up to 30 here: an entry one unit of the last place off (rotations whose products are not
    rounded alike: about one row of 2^16) has another weight."""
    from nano_vllm_amd import ops_seq
    H, seqs, T, page = 32, 128, 256, 128                   # a million (query, head)
    n, d = seqs * T, 128
    g = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn(n, H, 1, 2, generator=g, device="cuda").bfloat16().expand(n, H, 64, 2).reshape(n, H * d)
    kc = torch.zeros(3, page, 1, d, dtype=torch.bfloat16, device="cuda")        # page 0: the keys that show; 1 and 2: the portions' own
    vc = torch.zeros(3, 1, d, page, dtype=torch.bfloat16, device="cuda")
    kc[0, :, 0] = 8 * torch.eye(128, device="cuda")
    vc[0, 0] = torch.eye(128, device="cuda")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    por = ops_seq.Portions(i32([T * i for i in range(seqs + 1)]), i32([page] * seqs), i32(list(range(seqs))), torch.arange(seqs).repeat_interleave(T).to(torch.int32).cuda(), seqs, n, T)
    freq = torch.full((64,), 0.37, device="cuda")
    out = torch.empty(n, H * d, dtype=torch.bfloat16, device="cuda")
    ops_seq.window_attn(q, None, 1e-6, None, kc.view(-1, 1, d), vc.view(-1, 1, d), i32([[0, 1, 2]] * seqs), page, por, H, 1, d, d, 1.0, 0, out, rot_freq=freq)
    pairs = out.view(-1, 64, 2)
    assert not bool(torch.isnan(pairs).any()) and bool((pairs > 0).any())
    apart = (pairs != pairs[:, :1]).any(-1).any(-1).sum().item()
    assert apart == 0, f"{apart} of {n * H} rows"
