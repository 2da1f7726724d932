"""All layers of a small decode step in one launch (nvl_decode_step): against the step in float64 on the same 16-bit inputs, at the edges of its cuts (chunks of 32 keys, at most 30, 28, 24
and 24 parts in all, batches of 128 keys) and of its shapes; with its shares dealt instead of fixed; and what keeps the layers' own calls."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
W = 1024


def rand(g, *s, scale=1.0):
    return (scale * torch.randn(*s, generator=g, device="cuda")).bfloat16()


def step_inputs(lens, hq=16, ff=3072, layers=2, block=256, norms=True, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    hkv = hq // 2
    need = [max(1, -(-n // block)) for n in lens]
    table = torch.full((len(lens), max(need)), -1, dtype=torch.int32)
    ids = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)).to(torch.int32)
    at = 0
    for i, n in enumerate(need):
        if lens[i] > 0:
            table[i, :n] = ids[at:at + n]
        at += n
    every = []
    for _ in range(layers):
        norm = lambda n: (1 + 0.1 * torch.randn(n, generator=g, device="cuda")).bfloat16()
        cache = [rand(g, sum(need), hkv, block, 128) for _ in range(2)]
        for i, n in enumerate(lens):               # what a page holds behind the context, its new token's place among it, need not be finite
            if n > 0 and n % block:
                for c in cache:
                    c[table[i, (n - 1) // block], :, n - 1 - (n - 1) // block * block:] = float("nan")
        every.append((norm(W), rand(g, (hq + 2 * hkv) * 128, W, scale=W ** -0.5), norm(128) if norms else None, norm(128) if norms else None,
                      rand(g, W, hq * 128, scale=(hq * 128) ** -0.5), norm(W), rand(g, 2 * ff, W, scale=W ** -0.5), rand(g, W, ff, scale=ff ** -0.5), *cache))
    f = 1e6 ** (-torch.arange(0, 128, 2, dtype=torch.float64) / 128)
    ang = torch.arange(8192, dtype=torch.float64)[:, None] * f
    cs = torch.cat([ang.cos(), ang.sin()], 1).float().cuda()
    return rand(g, len(lens), W), every, cs, table.cuda(), torch.tensor(lens, dtype=torch.int32).cuda(), ff, hq


def exact(x, layers, cs, table, lens, ff, hq, block):
    """(last layer's output, residual, new keys and values of every layer) in float64."""
    def rms(v, w):
        return v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-6) * w.double()
    v, news = x.double(), []
    hkv = hq // 2
    for n1, wqkv, qn, kn, wo, n2, wgu, wd, kc, vc in layers:
        z = rms(v, n1) @ wqkv.double().T
        att, new = torch.zeros(len(v), hq * 128, dtype=torch.float64, device="cuda"), []
        for b, n in enumerate(lens.tolist()):
            if n <= 0:
                new.append(None)
                continue
            def turn(t, w):
                t = t.view(-1, 128)
                if w is not None:
                    t = rms(t, w)
                c, s = cs[n - 1, :64].double(), cs[n - 1, 64:].double()
                return torch.cat([t[:, :64] * c - t[:, 64:] * s, t[:, 64:] * c + t[:, :64] * s], 1)
            q, k, val = turn(z[b, :hq * 128], qn), turn(z[b, hq * 128:(hq + hkv) * 128], kn), z[b, (hq + hkv) * 128:].view(hkv, 128)
            new.append((k, val))
            pos = torch.arange(n - 1, device="cuda")
            blk = table[b, pos // block].long()
            ks = torch.cat([kc[blk, :, pos % block].double(), k[None]]).repeat_interleave(2, 1)
            vs = torch.cat([vc[blk, :, pos % block].double(), val[None]]).repeat_interleave(2, 1)
            p = torch.softmax((ks * q).sum(-1) * 128 ** -0.5, 0)
            att[b] = (p[..., None] * vs).sum(0).flatten()
        v1 = v + att @ wo.double().T
        gu = rms(v1, n2) @ wgu.double().T
        y = (torch.nn.functional.silu(gu[:, :ff]) * gu[:, ff:]) @ wd.double().T
        v = v1 + y
        news.append(new)
    return y, v1, news


def rel(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("lens,hq,ff,block,norms", [
    ([1], 16, 3072, 256, True), ([32], 16, 3072, 256, True), ([33], 16, 3072, 16, False), ([960], 16, 3072, 256, True), ([961], 16, 3072, 256, True),
    ([3841], 16, 3072, 256, True), ([7777], 8, 1024, 256, True), ([448, 449], 16, 3072, 256, True), ([0, 64], 16, 2048, 48, True), ([1800, 2], 8, 3072, 256, False),
    ([256, 257, 1], 16, 3072, 256, True), ([31, 0, 2100], 8, 2048, 32, True), ([192, 193, 768, 1537], 16, 3072, 256, True), ([1, 2, 3, 4], 16, 1024, 256, True),
    ([0, 0, 0, 5], 8, 1024, 256, True),
    ([3000, 40, 1, 700], 16, 3072, 256, True), ([33, 2500], 8, 1024, 64, True), ([0, 1500, 64], 16, 1024, 256, False)])
@pytest.mark.parametrize("patience", [200, 0])
def test_step(lens, hq, ff, block, norms, patience):
    """patience 0: the shares are dealt."""
    from nano_vllm_amd import ops
    x, layers, cs, table, ctx, ff, hq = step_inputs(lens, hq, ff, 2, block, norms, seed=len(lens) + sum(lens))
    want, v1, news = exact(x, layers, cs, table, ctx, ff, hq, block)
    before = [(l[8].clone(), l[9].clone()) for l in layers]
    out, residual = ops.decode_step(x, layers, 1e-6, cs, table, ctx, ff, hq, 128 ** -0.5, patience=patience)
    assert out.shape == (1, len(lens), W) and out.dtype == torch.float32
    # about eight roundings to 8 bits a layer on the way, 2^-9 / sqrt(3) each: 0.0045 over two layers
    assert rel(out[0], want) <= 2.0 ** -7 and rel(residual, v1) <= 2.0 ** -7
    for l, layer in enumerate(layers):             # the new token's key and value, and nothing else
        for b, n in enumerate(lens):
            if n > 0:
                blk, at = int(table[b, (n - 1) // block]), (n - 1) % block
                for i in range(2):
                    assert rel(layer[8 + i][blk, :, at], news[l][b][i]) <= 2.0 ** -7
                    before[l][i][blk, :, at] = layer[8 + i][blk, :, at]
        for i in range(2):
            assert torch.equal(layer[8 + i].view(torch.int16), before[l][i].view(torch.int16))


@pytest.mark.parametrize("lens,hq", [([700], 16), ([3841], 16), ([7777], 8), ([16000], 16), ([3000, 1111], 16), ([2100, 31, 960], 16), ([4096, 100, 1500, 2000], 16),
                                     ([0, 8000], 16), ([1, 1, 1, 6000], 16), ([1000, 1000, 4000, 1000], 16), ([5000, 0, 33, 65], 8), ([32, 6144, 32], 8)])
@pytest.mark.parametrize("patience", [200, 0])
def test_every_chunk_of_keys_counts(lens, hq, patience):
    """One layer whose attention is all there is to see: queries are sqrt(128) in entry 0 alone (no rotation), and so are the first and the last key of every chunk of 32 and the new token's;
    other keys are 0, so the weights lie on those, all alike. The i-th of them shows in entry i % 128 of the result with 1 + i // 128; o hands eight heads on as they are. A key that is
    left out, or counts twice, moves its entry by 2.6 % at least (eight keys of 1 to 8 in one), the bound is 0.8 %."""
    from nano_vllm_amd import ops
    block, W8 = 256, min(hq, 8) * 128
    x, layers, cs, table, ctx, ff, hq = step_inputs(lens, hq, 1024, 1, block, True, seed=7)
    n1, wqkv, qn, kn, wo, n2, wgu, wd, kc, vc = layers[0]
    cs, hkv = cs[:1].expand(16384, 128).contiguous(), hq // 2       # position 0's angles everywhere
    for t in (x, wqkv, wo, kc, vc):
        t.zero_()
    for t in (n1, qn, kn):
        t.fill_(1)
    wo[:W8, :W8] = torch.eye(W8, device="cuda")
    want = torch.zeros(len(lens), 128, dtype=torch.float64)
    for row, n in enumerate(lens):
        if n == 0:
            continue
        x[row, row] = 1.0                          # the norm makes 32 of it; its column of the projection is the row's query, key and value
        keys = sorted({k for c in range(0, n, 32) for k in (c, min(c + 31, n - 1))})
        blk, at = table[row, torch.tensor(keys[:-1], dtype=torch.long) // block].long(), torch.tensor(keys[:-1], dtype=torch.long, device="cuda") % block
        entry, value = torch.arange(len(keys)) % 128, 1.0 + torch.arange(len(keys)) // 128
        kc[blk, :, at, 0] = 128 ** 0.5
        vc[blk, :, at, entry[:-1].cuda()] = value[:-1, None].bfloat16().cuda()
        wqkv[:(hq + hkv) * 128:128, row] = 1.0
        wqkv[(hq + hkv) * 128 + int(entry[-1])::128, row] = float(value[-1]) / 32
        want[row].index_add_(0, entry, value.double() / (len(keys) + (n - len(keys)) * math.exp(-128 ** 0.5)))
    out, residual = ops.decode_step(x, layers, 1e-6, cs, table, ctx, ff, hq, 128 ** -0.5, patience=patience)
    for h in range(min(hq, 8)):
        got = residual[:, h * 128:(h + 1) * 128].double().cpu() - x[:, h * 128:(h + 1) * 128].double().cpu()
        # the result and (where the row's 1 stands) the residual are rounded to 8 bits; the new token's value, weights and scores by less than 2^-8 more
        bound = want * 2.0 ** -7 + x[:, h * 128:(h + 1) * 128].double().cpu() * 2.0 ** -7
        assert bool(((got - want).abs() <= bound).all()), (h, ((got - want).abs() - bound).max())


@pytest.mark.parametrize("lens", [[700], [5, 900], [1, 300, 1500], [300, 31, 900, 2000]])
def test_dealt_shares_give_the_same_bits_and_so_do_replays(lens):
    from nano_vllm_amd import ops
    x, layers, cs, table, ctx, ff, hq = step_inputs(lens, layers=3)
    args = (x, layers, 1e-6, cs, table, ctx, ff, hq, 128 ** -0.5)
    ws = torch.zeros(ops.decode_step_bytes(len(lens), 3, W, ff, hq, hq // 2) // 4, dtype=torch.int32, device="cuda")
    fixed = ops.decode_step(*args, patience=1 << 20, workspace=ws)        # (all of them are seen long before)
    assert int(ws[1]) == 1 and int(ws[0]) == 256 and int(ws[2]) == 0      # the sync words: all came, no share was dealt
    dealt = ops.decode_step(*args, patience=0, workspace=ws)
    hkv, parts = hq // 2, min(32, (256 - len(lens) * hq) // (len(lens) * hq // 2))
    assert int(ws[1]) == 2 and int(ws[2]) == 3 * ((hq + 2 * hkv) * 8 + len(lens) * hkv * parts + len(lens) * hq + 3 * 256) + 256        # every share, and one more look of each workgroup
    assert torch.equal(fixed[0], dealt[0]) and torch.equal(fixed[1], dealt[1])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = ops.decode_step(*args)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(held[0], fixed[0]) and torch.equal(held[1], fixed[1])
        held[0].zero_()
        again = ops.decode_step(*args)
        assert torch.equal(again[0], fixed[0])


@pytest.mark.parametrize("patience", [200, 0])
@pytest.mark.parametrize("asks", [0, 1, 8])
def test_a_step_that_gives_up_says_so_and_stores_no_row_that_is_not_its_own(asks, patience):
    """Waits that end early leave NaN, the word, and in the caches nothing but rows of the new token's own."""
    from nano_vllm_amd import ops
    lens = [700, 40, 257]
    x, layers, cs, table, ctx, ff, hq = step_inputs(lens, layers=3)
    args = (x, layers, 1e-6, cs, table, ctx, ff, hq, 128 ** -0.5)
    before = [(l[8].clone(), l[9].clone()) for l in layers]
    word = torch.zeros(1, dtype=torch.int32, device="cuda")
    out, residual = ops.decode_step(*args, patience=patience, asks=asks, gave_up=word)
    gave = int(word)
    early = [(l[8].clone(), l[9].clone()) for l in layers]
    want, kept = ops.decode_step(*args, gave_up=word)
    assert int(word) == gave and (asks or gave)     # (a step that did not give up leaves the word as it is)
    for got, right in ((out, want), (residual, kept)):
        assert bool((got == right).all()) or gave and bool((got.isnan() | (got == right)).all())
    for l, layer in enumerate(layers):             # every row is as it was or the step's
        for i in range(2):
            rows = torch.stack([c.view(torch.int16) for c in (early[l][i], before[l][i], layer[8 + i])])
            same = (rows[0] == rows[1]).all(-1)
            assert bool((same | (rows[0] == rows[2]).all(-1)).all())
    assert asks or out.isnan().any()               # (no workgroup is as fast as its first look in all of 18 phases)


def test_the_engine_raises_where_a_step_gave_up(tmp_path, monkeypatch):
    import json
    from nano_vllm_amd import LLM, SamplingParams, ops
    (tmp_path / "config.json").write_text(json.dumps(dict(
        architectures=["Qwen3ForCausalLM"], model_type="qwen3", hidden_size=1024, intermediate_size=1024, num_hidden_layers=2, num_attention_heads=8, num_key_value_heads=4, head_dim=128,
        rms_norm_eps=1e-6, vocab_size=512, hidden_act="silu", max_position_embeddings=2048, rope_theta=1e6, tie_word_embeddings=True, attention_bias=False, torch_dtype="bfloat16")))
    llm = LLM(str(tmp_path), dummy_weights=True, enforce_eager=True, max_model_len=512, num_kvcache_blocks=16, max_num_seqs=8)
    try:
        ran, calls = ops.decode_step, []
        monkeypatch.setattr(ops, "decode_step", lambda *a, **k: (calls.append(1), ran(*a, **k))[1])
        ask = lambda: llm.generate([[1, 2, 3], [4, 5]], SamplingParams(temperature=0.0, max_tokens=6, ignore_eos=True), use_tqdm=False)
        assert [len(o["token_ids"]) for o in ask()] == [6, 6] and calls
        monkeypatch.setattr(ops, "decode_step", lambda *a, **k: ran(*a, **dict(k, asks=0)))
        with pytest.raises(ops.NvlError, match="gave up"):
            ask()
        monkeypatch.setattr(ops, "decode_step", ran)
        with pytest.raises(ops.NvlError, match="gave up"):       # its rows are still missing
            ask()
        torch.cuda.synchronize()
    finally:
        llm.exit()


def test_a_row_that_is_no_number_stays_its_own():
    from nano_vllm_amd import ops
    x, layers, cs, table, ctx, ff, hq = step_inputs([40, 500, 33])
    clean = ops.decode_step(x, layers, 1e-6, cs, table, ctx, ff, hq, 128 ** -0.5)[0].clone()
    bad = x.clone()
    bad[1, 7] = float("nan")
    bad.view(torch.int16)[1, 8] = -1               # the word that means "not written", as a NaN of the input
    got = ops.decode_step(bad, layers, 1e-6, cs, table, ctx, ff, hq, 128 ** -0.5)[0]
    assert got[0, 1].isnan().all() and torch.equal(got[0, [0, 2]], clean[0, [0, 2]])


def test_what_is_not_covered_is_refused():
    from nano_vllm_amd import ops
    assert ops.decode_step_bytes(4, 28, 1024, 3072, 16, 8) > 0
    for shape in [(5, 28, 1024, 3072, 16, 8), (0, 28, 1024, 3072, 16, 8), (1, 41, 1024, 3072, 16, 8), (1, 28, 2048, 6144, 16, 8), (1, 28, 1024, 4096, 16, 8),
                  (1, 28, 1024, 3072, 16, 16), (1, 28, 1024, 3072, 32, 16)]:
        assert ops.decode_step_bytes(*shape) == 0
    x, layers, cs, table, ctx, ff, hq = step_inputs([3] * 5)
    with pytest.raises(ops.NvlError, match="rows"):
        ops.decode_step(x, layers, 1e-6, cs, table, ctx, ff, hq, 128 ** -0.5)


@pytest.mark.parametrize("touch", ["nothing", "layer", "attention", "mlp", "norm", "projection", "global", "own call", "rows", "context", "refused"])
def test_calls_that_somebody_watches_are_made(touch, monkeypatch):
    from nano_vllm_amd import ops, qwen3
    from nano_vllm_amd.attn_meta import reset_context, set_context
    from types import SimpleNamespace
    config = SimpleNamespace(hidden_size=1024, intermediate_size=1024, num_hidden_layers=2, num_attention_heads=8, num_key_value_heads=4, head_dim=128, rms_norm_eps=1e-6,
                             vocab_size=512, hidden_act="silu", max_position_embeddings=8192, rope_theta=1e6, tie_word_embeddings=True, attention_bias=False)
    torch.manual_seed(1)
    torch.set_default_dtype(torch.bfloat16)
    torch.set_default_device("cuda")
    try:
        model = qwen3.Qwen3ForCausalLM(config)
        for p in model.parameters():
            p.data.copy_(1 + 0.1 * torch.randn(p.shape) if p.dim() == 1 else torch.randn(p.shape) * p.shape[-1] ** -0.5)
    finally:
        torch.set_default_device("cpu")
        torch.set_default_dtype(torch.float32)
    rows = 5 if touch == "rows" else 2
    for m in model.modules():
        if isinstance(m, qwen3.Attention):
            m.k_cache, m.v_cache = (torch.randn(rows, 4, 256, 128, device="cuda").bfloat16() for _ in range(2))
    layer, seen, calls, width = model.model.layers[1], [], [], 40 if touch == "context" else 1
    watched = {"layer": layer, "attention": layer.self_attn, "mlp": layer.mlp, "norm": layer.post_attention_layernorm, "projection": layer.self_attn.o_proj}
    hook = lambda *a: seen.append(1)
    handle = watched[touch].register_forward_hook(hook) if touch in watched else None
    if touch == "global":
        handle = torch.nn.modules.module.register_module_forward_hook(hook)
    if touch == "own call":
        inner = layer.mlp.forward
        layer.mlp.forward = lambda *a, **k: (seen.append(1), inner(*a, **k))[1]
    ran = ops.decode_step
    monkeypatch.setattr(ops, "decode_step", lambda *a, **k: (calls.append(1), ran(*a, **k))[1])
    ids, pos = torch.arange(rows).cuda(), torch.full((rows,), 99).cuda()

    def step():
        set_context(False, slot_mapping=None, context_lens=torch.full((rows,), 100, dtype=torch.int32).cuda(),
                    block_tables=torch.nn.functional.pad(torch.arange(rows, dtype=torch.int32).cuda()[:, None], (0, width - 1), value=-1),
                    max_context=width * 256 if touch != "refused" else 512)
        out = model(ids, pos)
        reset_context()
        return out
    try:
        with torch.inference_mode():
            if touch == "refused":               # a block table too narrow, as before
                with pytest.raises(ops.NvlError, match="narrower"):
                    step()
                return
            got = step()
            monkeypatch.setattr(qwen3, "_DECODE_STEP", False)
            apart = step()
    finally:
        if handle is not None:
            handle.remove()
    assert bool(calls) == (touch == "nothing")
    assert rel(got, apart.double()) <= 2.0 ** -6   # two ways of two layers' roundings
