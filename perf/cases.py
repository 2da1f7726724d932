"""The work this framework is used for, as measurable cases: one step of a served model — a batch of prompts, or one decoded
token for every running sequence — for the transformer family of the benchmark (paged K/V of 128-wide heads) and for the six
families of the model registry whose layers are listed in config.json (windowed, block-masked, latent and pooled attention,
recurrences, routed experts). Sizes are those of bench.py (its 256-sequence workload, its long prompts, and `--compare-families`).

A case: model `family`, its `size` (a name of the weights module for qwen3, the width for the others), `step` ("prompts": every
sequence brings a whole prompt, or, behind `cached` tokens that are in the pages already, the rest of one; "decode": every sequence
brings one token), `seqs` sequences of `lo` to `hi` tokens (prompt lengths, or contexts of a decode step), and the activation `dtype`.

A step is run as the engine runs it: step metadata through set_context, the model's forward, compute_logits; prompts eagerly, a
decode step as the replay of a captured graph. Weights are seeded random tensors of a trained model's magnitudes: matrices scaled by
their fan-in, norms around one, and embeddings that say nothing along the routers' rows but which experts are their token's, so that a
token's experts are chosen by a margin and not by the last bit (as a trained router's are).
"""
import json
import math
import os
import random
import tempfile
import zlib

import torch

VOCAB = 32768                     # of the registry's families, as in bench.py --compare-families
PAGE = 256
FAMILIES = ("foduzen", "nokipel", "pefazen", "lobidra", "ligidra", "reselorn")
F64 = torch.float64


def listed():
    def case(name, family, size, step, seqs, lo, hi, cached=0, dtype="bfloat16"):
        return dict(name=name, family=family, size=size, step=step, seqs=seqs, lo=lo, hi=hi, cached=cached, dtype=dtype)
    return [
        # interactive use: one user waiting for the next token
        case("qwen3 decode, one sequence", "qwen3", "qwen3-0.6b", "decode", 1, 700, 700),
        # the reference's benchmark in the middle of its run: 256 sequences, contexts as its prompts and outputs make them
        case("qwen3 decode, 256 sequences", "qwen3", "qwen3-0.6b", "decode", 256, 100, 2047),
        # its prompt steps: as many prompts of 100 to 1,024 tokens as fill a step
        case("qwen3 prompts", "qwen3", "qwen3-0.6b", "prompts", 26, 100, 1024),
        # long documents that arrive in portions: the rest of each prompt attends to the part in the pages
        case("qwen3 long prompts, cached", "qwen3", "qwen3-8b-2l", "prompts", 2, 6000, 8191, cached=4096),
        # a full prompt step of the other families, ragged as users' prompts are
        case("foduzen prompts", "foduzen", 4096, "prompts", 9, 1100, 2048),
        case("nokipel prompts", "nokipel", 4096, "prompts", 9, 1100, 2048),
        case("pefazen prompts", "pefazen", 1024, "prompts", 9, 1100, 2048),
        case("lobidra prompts", "lobidra", 1024, "prompts", 9, 1100, 2048),
        case("ligidra prompts", "ligidra", 4096, "prompts", 9, 1100, 2048),
        # serving traffic once the prompts are in: 64 sequences, one token each
        case("nokipel decode", "nokipel", 1024, "decode", 64, 200, 1500),
        case("reselorn decode", "reselorn", 4096, "decode", 64, 200, 1500),
        # a few short requests in full precision, as evaluations run them
        case("ligidra short prompts, float32", "ligidra", 1024, "prompts", 3, 20, 200, dtype="float32"),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    step = rng.choice(("prompts", "decode"))
    if rng.random() < 0.3:
        family, size = "qwen3", rng.choice(("qwen3-0.6b", "qwen3-8b-2l"))
    else:
        family, size = rng.choice(FAMILIES), rng.choice((1024, 2048, 4096))
    dtype = "float32" if family != "qwen3" and size == 1024 and rng.random() < 0.2 else "bfloat16"
    cached = 0
    if step == "decode":
        seqs = log_int(1, 256 if family == "qwen3" else 64)
        hi = log_int(64, 2047 if family == "qwen3" else 1500)
    else:
        most = 512 if dtype == "float32" else 14000
        hi = log_int(16, min(most, 8000 if family == "qwen3" else 3000))
        seqs = log_int(1, max(1, min(32, most // hi)))
        if family == "qwen3" and rng.random() < 0.4:
            cached = PAGE * rng.randint(1, 12)
    lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
    return dict(family=family, size=size, step=step, seqs=seqs, lo=lo, hi=hi, cached=cached, dtype=dtype)


# ---- sizes ---------------------------------------------------------------------------------------------------------------
def _lens(case):
    r = random.Random(f"{case['seqs']} {case['lo']} {case['hi']}")
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["seqs"])]


def _config(case):
    """The parsed config.json of a registry family: layers of a real model's size (bench.py --compare-families)."""
    W = case["size"]
    ff, heads, kv, layers = 3 * W, 32 if W == 4096 else 16, 8, 4 if W == 1024 else 2
    att = {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5}
    moe = {"kind": "moe", "expert": {"ff": ff // 4}, "shared": {"ff": ff // 4}, "router": {"experts": 32, "top": 4}}
    dense = {"kind": "dense", "ff": ff}
    bands = {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 2048}
    yarn = {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}
    raw = {"norm": {"eps": 1e-6}, "vocab": VOCAB, "width": W, "embedding": {"scale": 1.0}}
    out, nh = [], W // 128
    for i in range(layers):
        odd = i % 2 == 1
        if case["family"] == "foduzen":
            out.append({"type": "rglru", "mlp": dense, "mixer": {"width": W, "blocks": nh, "conv": 4}} if odd else
                       {"type": "parallel", "mlp": dense,
                        "mixer": {"left": dict(att, mask={"size": 1024}),
                                  "right": {"heads": W // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}}})
        elif case["family"] == "nokipel":
            raw["norm"]["groups"] = 1
            routed = {"kind": "moe", "expert": {"ff": ff // 4}, "shared": {"ff": ff // 4},
                      "router": {"experts": 30, "identity": 2, "top": 3, "scale": 1.0, "groups": {"count": 4, "keep": 2}}}
            out.append({"type": "lightning", "mlp": dict(dense, limit=7.0),
                        "mixer": {"heads": nh, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** (-3 - 5 * j / max(nh - 1, 1)) for j in range(nh)]}}
                       if odd else {"type": "attention", "mixer": dict(att, mask={"size": 1024}, rot={"dims": 64, "base": 500000.0}), "mlp": routed})
        elif case["family"] == "pefazen":
            raw.update(residual_mult=1.0, logit_scale=1.0, logit_softcap=30.0)
            m = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 3 * W // 8, "kv_rank": 192, "scale": 192 ** -0.5}
            if odd:
                m["rot"] = {"dims": 64, "base": 500000.0, "scaling": dict(yarn, factor=8.0)}
            else:
                m.update(mask={"size": 1024}, rot={"dims": 64, "base": 10000.0}, **({"kv_from": 0} if i == 2 else {}))
            out.append({"type": "latent_attention_2" if odd else "latent_attention", "mixer": m,
                        "mlp": {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 32, "top": 4}}})
        elif case["family"] == "lobidra":
            layer = {"type": "parallel", "mlp": dense,
                     "mixer": {"left": dict(att, q_temp={"coef": 0.1, "every": 1024}),
                               "right": {"heads": nh, "dim": 128, "vdim": 128, "gate_cap": 15.0}, "left_scale": 0.7, "right_scale": 0.7}} if odd else \
                    {"type": "attention", "mixer": dict(att, conv=4, rot={"dims": 64, "base": 500000.0, "scaling": bands}), "mlp": moe}
            out.append(dict(layer, weights_of=i % 2) if i >= 2 else layer)
        elif case["family"] == "ligidra":
            raw["token_side"] = {"dim": W // 16}
            out.append({"type": "channel_delta" if i % 4 == 1 else "delta", "mlp": moe,
                        "mixer": {"heads": nh, "kv_heads": nh // 2, "dim": 128, "vdim": 128, "conv": 4}} if odd else
                       {"type": "attention", "mlp": moe, "mixer": dict(att, softcap=30.0, mask={"size": 1024, "pool": 16},
                                                                       rot={"dims": 64, "base": 500000.0, "scaling": bands}, **({"kv_from": 0} if i else {}))})
        else:
            out.append({"type": "attention", "mlp": moe if odd else dense,
                        "mixer": dict(att, mask={"size": 1024}, v_mix=True, rot={"dims": 64, "base": 500000.0, "scaling": yarn})})
    raw.update(architecture=case["family"].capitalize(), layers=out)
    return raw


def _qwen3(case):
    from nano_vllm_amd.weights import qwen3_config_dict
    return qwen3_config_dict(case["size"])


# ---- weights and inputs, from the seed alone -----------------------------------------------------------------------------
class _Weights:
    """Checkpoint tensors by name, made on the GPU: values that bfloat16 holds exactly."""

    def __init__(self, case, seed, raw):
        self.family, self.seed, self.raw, self.leanings = case["family"], int(seed), raw, None

    def gen(self, name):
        return torch.Generator(device="cuda").manual_seed((self.seed << 32) ^ zlib.crc32(name.encode()))

    def randn(self, name, shape):
        return torch.randn(shape, generator=self.gen(name), dtype=torch.float32, device="cuda")

    def directions(self):
        """For every routed layer the rows of its router (orthonormal), and for every token a step along those of its experts."""
        if self.leanings is None:
            W, rows, steps = self.raw["width"], {}, []
            routed = [i for i, layer in enumerate(self.raw["layers"]) if "router" in (layer.get("mlp") or {}) and self.family != "lobidra"]
            total = [self.raw["layers"][i]["mlp"]["router"] for i in routed]
            total = [r["experts"] + r.get("identity", 0) for r in total]
            if routed:
                basis = torch.linalg.qr(self.randn("router.basis", (W, sum(total))))[0].T.contiguous()
                at = 0
                for i, n in zip(routed, total):
                    r = self.raw["layers"][i]["mlp"]["router"]
                    g = (r.get("groups") or {"count": 1})["count"]
                    u = torch.rand((VOCAB, n), generator=self.gen(f"experts.{i}"), dtype=torch.float32, device="cuda")
                    if g > 1:              # two experts of one group, the others of a second one
                        keep = torch.rand((VOCAB, g), generator=self.gen(f"groups.{i}"), dtype=torch.float32, device="cuda").argsort(1)[:, :2]
                        u = u.view(VOCAB, g, n // g)
                        order = u.argsort(2)
                        first = keep[:, 0] * (n // g) + order[torch.arange(VOCAB, device="cuda"), keep[:, 0], 0]
                        again = keep[:, 0] * (n // g) + order[torch.arange(VOCAB, device="cuda"), keep[:, 0], 1]
                        other = keep[:, 1] * (n // g) + order[torch.arange(VOCAB, device="cuda"), keep[:, 1], 0]
                        mine = torch.stack([first, again, other], 1)
                    else:
                        mine = u.argsort(1)[:, :r["top"]]
                    z = torch.full((VOCAB, n), -6.0 * mine.shape[1] / n, dtype=torch.float32, device="cuda")
                    z.scatter_(1, mine, 6.0 * (1.0 - mine.shape[1] / n))
                    steps.append(z)
                    rows[i] = basis[at:at + n]
                    at += n
                self.leanings = rows, (torch.cat(steps, 1), basis)
            else:
                self.leanings = rows, None
        return self.leanings

    def __call__(self, name, *shape):
        parts, leaf, fam = name.split("."), name.split(".")[-1], self.family
        if leaf == "table":                                  # a row: distinct experts of the token
            n = self.raw["layers"][int(parts[0][1:])]["mlp"]["router"]["experts"]
            return torch.rand((shape[0], n), generator=self.gen(name), dtype=torch.float32, device="cuda").argsort(1)[:, :shape[1]].to(torch.int32)
        if leaf == "router":
            return self.directions()[0][int(parts[0][1:])].to(torch.bfloat16)
        t = self.randn(name, shape)
        offset_norms = fam == "lobidra" and "right" not in parts
        if fam == "qwen3":
            t = 1.0 + 0.1 * t if len(shape) == 1 else t / shape[-1] ** 0.5 * (shape[-1] ** 0.5 if "embed" in name else 0.5 if "down" in name else 1.0)
        elif name == "embed":
            if self.directions()[1] is not None:             # nothing but the steps along the routers' rows
                steps, basis = self.directions()[1]
                t = t + (steps - t @ basis.T) @ basis
        elif name == "side.embed" or leaf == "sink":
            pass
        elif "side" in parts and leaf == "norm":
            t = 0.2 + 0.02 * t
        elif leaf in ("norm", "norm1", "norm2", "norm1b", "norm2b", "out", "D"):
            t = 0.1 * t + (0.0 if offset_norms else 1.0)
            if leaf in ("norm1b", "norm2b"):                 # a branch enters the stream at about half its size
                t = t - 0.5
            elif fam == "foduzen" and leaf in ("norm1", "norm2"):
                t = 0.5 * t
        elif leaf in ("ls1", "ls2"):
            t = 0.3 + 0.05 * t
        elif leaf == "vmix" or leaf == "shift":
            t = torch.sigmoid(t)
        elif leaf == "lam":
            t = -3.5 + 0.8 * t
        elif leaf == "A_log":
            t = -1.0 + 0.7 * t
        elif leaf == "dt_bias":
            t = -2.0 + t
        elif leaf == "act":
            t = 0.5 * t
        elif leaf == "correction":
            t = 0.02 * t
        elif leaf == "b" and not (fam == "ligidra" and len(shape) == 2):
            t = (t + (2.0 if name.endswith("f.b") else 0.0)) if fam == "lobidra" else 0.1 * t
        else:
            t = t / (shape[-1] if shape else 1) ** 0.5 * ((0.2 if fam == "pefazen" else 0.4) if leaf == "down" else 1.0)
        return t.to(torch.bfloat16)


def _tokens(case, seed, vocab):
    g = torch.Generator(device="cuda").manual_seed((int(seed) << 32) ^ 0x70AE)
    n = sum(_lens(case))
    return torch.randint(0, vocab, (n,), generator=g, device="cuda")


def _page_table(lens, seed):
    """Scattered page ids [seqs, most pages] (-1: none) of sequences of `lens` tokens, and how many pages there are."""
    need = [-(-n // PAGE) for n in lens]
    ids = list(range(sum(need)))
    random.Random(int(seed)).shuffle(ids)
    table, at = torch.full((len(lens), max(need)), -1, dtype=torch.int32), 0
    for i, k in enumerate(need):
        table[i, :k] = torch.tensor(ids[at:at + k], dtype=torch.int32)
        at += k
    return table, len(ids)


def _cached_kv(case, seed, layer, pages, kv_heads):
    """Keys and values an earlier step left in the pages of a layer: [pages, kv heads, PAGE, 128] each."""
    g = torch.Generator(device="cuda").manual_seed((int(seed) << 32) ^ zlib.crc32(f"kv.{layer}".encode()))
    return [torch.randn((pages, kv_heads, PAGE, 128), generator=g, dtype=torch.bfloat16, device="cuda") for _ in range(2)]


# ---- the step ------------------------------------------------------------------------------------------------------------
def _build(case, seed):
    """(model with its weights, parsed configuration) as a serving program makes them."""
    from nano_vllm_amd.registry import resolve
    raw = _qwen3(case) if case["family"] == "qwen3" else _config(case)
    with tempfile.TemporaryDirectory() as path:
        with open(os.path.join(path, "config.json"), "w") as fh:
            json.dump(raw, fh)
        spec, config = resolve(path)
    dtype = getattr(torch, case["dtype"])
    config.kvcache_block_size = PAGE
    before = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    torch.set_default_device("cuda")
    try:
        with torch.inference_mode():
            model = spec.build(config, dtype)
            weights = _Weights(case, seed, raw)
            if case["family"] == "qwen3":
                from nano_vllm_amd.weights import parameter_shapes
                for name, shape in parameter_shapes(raw).items():
                    for part, (fused, shard) in model.packed_modules_mapping.items():
                        if part in name:
                            p = model.get_parameter(name.replace(part, fused))
                            p.weight_loader(p, weights(name, *shape), shard)
                            break
                    else:
                        p = model.get_parameter(name)
                        p.weight_loader(p, weights(name, *shape)) if hasattr(p, "weight_loader") else p.data.copy_(weights(name, *shape))
                for m in model.modules():
                    if hasattr(m, "pack_for_decode"):
                        m.pack_for_decode()
            else:
                shapes = __import__(f"nano_vllm_amd.{case['family']}", fromlist=["tensor_shapes"]).tensor_shapes(raw)
                loaders = model.named_loaders()
                for name, shape in shapes.items():
                    loaders[name](weights(name, *shape))
    finally:
        torch.set_default_device("cpu")
        torch.set_default_dtype(before)
    return model, raw


def _captured(step):
    """`step` as a graph: (replay, its outputs)."""
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


@torch.inference_mode()
def prepare(case, seed):
    model, raw = _build(case, seed)
    prepared = _prepare_qwen3 if case["family"] == "qwen3" else _prepare_packed
    return prepared(case, seed, model, raw)


def _prepare_qwen3(case, seed, model, raw):
    from nano_vllm_amd import ops
    from nano_vllm_amd.attn_meta import reset_context, set_context
    lens, cached, decode = _lens(case), case["cached"], case["step"] == "decode"
    heads, kv_heads = raw["num_attention_heads"], raw["num_key_value_heads"]
    table, pages = _page_table([n + cached for n in lens], seed)
    for i, m in enumerate(m for m in model.modules() if hasattr(m, "k_cache") and hasattr(m, "v_cache")):
        if decode or cached:
            m.k_cache, m.v_cache = _cached_kv(case, seed, i, pages, kv_heads)
        else:
            m.k_cache, m.v_cache = (torch.zeros((pages, kv_heads, PAGE, 128), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    ids = _tokens(case, seed, raw["vocab_size"])
    # a decode step's token is the last one of its sequence; the rest of the context is in the pages
    spans = [(n - 1, n) if decode else (cached, cached + n) for n in lens]
    pos = torch.cat([torch.arange(a, b) for a, b in spans])
    slots = torch.cat([table[i, torch.arange(a, b) // PAGE] * PAGE + torch.arange(a, b) % PAGE for i, (a, b) in enumerate(spans)])
    pos, slots, table = pos.cuda(), slots.to(torch.int32).cuda(), table.cuda()
    if decode:
        ids = ids[torch.tensor(lens).cumsum(0).sub(1).cuda()].clone()
        longest = 4096                                       # the engine's default max_model_len, which sizes the block table
        table = torch.nn.functional.pad(table, (0, longest // PAGE - table.shape[1]), value=-1)
        ctx = torch.tensor(lens, dtype=torch.int32, device="cuda")
        ws = torch.zeros(ops.paged_attn_decode_workspace_bytes(len(lens), heads, longest), dtype=torch.uint8, device="cuda")
        plan = torch.zeros(ops.decode_plan_bytes(), dtype=torch.uint8, device="cuda")

        def step():
            ops.decode_plan(ctx, heads, kv_heads, longest, plan)
            set_context(False, slot_mapping=slots, context_lens=ctx, block_tables=table, decode_workspace=ws, max_context=longest, decode_plan=plan)
            logits = model.compute_logits(model(ids, pos))
            reset_context()
            return logits
        graph, logits = _captured(step)
        return {"graph": graph, "logits": logits, "keep": (model, ids, pos, slots, table, ctx, ws, plan)}
    cu_q = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    cu_k = torch.tensor([0] + [n + cached for n in lens]).cumsum(0).to(torch.int32)
    args = (True, cu_q.cuda(), cu_k.cuda(), max(lens), max(lens) + cached, slots, None, table if cached else None)
    return {"model": model, "ids": ids, "pos": pos, "context": (args, {}), "rows": None}


def _prepare_packed(case, seed, model, raw):
    from nano_vllm_amd.attn_meta import reset_context, set_context
    from nano_vllm_amd.ops_seq import Portions
    lens, decode, dtype = _lens(case), case["step"] == "decode", getattr(torch, case["dtype"])
    table, pages = _page_table(lens, seed)
    states = []
    for m in model.modules():                                # pages and state slots, as the layers ask for them
        if hasattr(m, "kv_shapes") and m.kv_shapes() is not None:
            k, v = m.kv_shapes()
            m.k_cache = torch.zeros(pages * PAGE, *k, dtype=dtype, device="cuda")
            m.v_cache = torch.zeros(pages * PAGE, *v, dtype=dtype, device="cuda")
            m.block_size = PAGE
        if hasattr(m, "page_shapes"):
            for name, shape in m.page_shapes().items():
                setattr(m, name, torch.zeros(pages, *shape, dtype=dtype, device="cuda"))
        if hasattr(m, "state_shapes"):
            for name, shape in m.state_shapes().items():
                setattr(m, name, torch.zeros(len(lens) + 1, *shape, dtype=torch.float32, device="cuda"))
                states.append(getattr(m, name))
    ids = _tokens(case, seed, VOCAB)
    starts = torch.tensor([0] + lens).cumsum(0).tolist()
    gpu_table = table.cuda()

    def portions(which, spans):
        """Tokens [a, b) of the sequences `which` as one packed step."""
        pos = torch.cat([torch.arange(a, b) for a, b in spans])
        slots = torch.cat([table[i, torch.arange(a, b) // PAGE] * PAGE + torch.arange(a, b) % PAGE for i, (a, b) in zip(which, spans)])
        n = [b - a for a, b in spans]
        cu = torch.tensor([0] + n).cumsum(0).to(torch.int32)
        tseq = torch.repeat_interleave(torch.arange(len(which)), torch.tensor(n)).to(torch.int32)
        por = Portions(cu.cuda(), torch.tensor([a for a, _ in spans], dtype=torch.int32).cuda(), torch.tensor(which, dtype=torch.int32).cuda(),
                       tseq.cuda(), len(which), int(cu[-1]), max(n))
        tokens = torch.cat([ids[starts[i] + a:starts[i] + b] for i, (a, b) in zip(which, spans)])
        rows = (cu[1:] - 1).to(torch.int32).cuda()
        context = ((True,), dict(slot_mapping=slots.to(torch.int32).cuda(), block_tables=gpu_table[which].contiguous(), portions=por))
        return {"model": model, "ids": tokens, "pos": pos.cuda(), "context": context, "rows": rows}

    every = list(range(len(lens)))
    if not decode:
        return portions(every, [(0, n) for n in lens])
    batch, room = [], 16384                                  # everything but the last token of every sequence, in steps of at most 16,384
    for i in every + [None]:
        if batch and (i is None or lens[i] - 1 > room):
            run(portions(batch, [(0, lens[j] - 1) for j in batch]))
            batch, room = [], 16384
        if i is not None and lens[i] > 1:
            batch.append(i)
            room -= lens[i] - 1
    state = portions(every, [(n - 1, n) for n in lens])
    after_prompts = [s.clone() for s in states]

    def step():
        set_context(*state["context"][0], **state["context"][1])
        logits = model.compute_logits(model(state["ids"], state["pos"]), state["rows"], len(lens))
        reset_context()
        return logits
    graph, logits = _captured(step)
    for s, before in zip(states, after_prompts):
        s.copy_(before)
    return {"graph": graph, "logits": logits, "keep": (model, state, states)}


@torch.inference_mode()
def run(state):
    if "graph" in state:
        state["graph"].replay()
        return {"logits": state["logits"]}
    from nano_vllm_amd.attn_meta import reset_context, set_context
    model, rows = state["model"], state["rows"]
    set_context(*state["context"][0], **state["context"][1])
    hidden = model(state["ids"], state["pos"])
    logits = model.compute_logits(hidden) if rows is None else model.compute_logits(hidden, rows, rows.numel())
    reset_context()
    return {"logits": logits}


# ---- what a step cannot do without ---------------------------------------------------------------------------------------
def work(case):
    lens, cached, decode = _lens(case), case["cached"], case["step"] == "decode"
    n, esize = (len(lens) if decode else sum(lens)), 4 if case["dtype"] == "float32" else 2
    flops = nbytes = 0.0

    def keys(a, b, window=0, chunk=0):
        """Visible (query, key) pairs of the queries at positions [a, b)."""
        p = torch.arange(a, b, dtype=F64)
        return float((p % chunk + 1 if chunk else (p + 1).clamp(max=window) if window else p + 1).sum())
    spans = [(m - 1, m) if decode else (cached, cached + m) for m in lens]

    def attend(heads, d, dv, kv_heads, window=0, chunk=0, store=True):
        nonlocal flops, nbytes
        flops += sum(2.0 * heads * (d + dv) * keys(a, b, window, chunk) for a, b in spans)
        seen = sum(min(a, window - 1) if window else (a % chunk if chunk else a) for a, _ in spans)
        nbytes += (seen + (n if store else 0)) * kv_heads * (d + dv) * esize

    def dense(out, width):
        nonlocal flops, nbytes
        flops += 2.0 * n * out * width
        nbytes += out * width * esize

    def experts(E, top, ff, width, mats):
        nonlocal flops, nbytes
        flops += 2.0 * n * top * ff * width * mats
        nbytes += E * (1.0 - (1.0 - top / E) ** n) * ff * width * mats * esize

    def memory(heads, d, dv):
        nonlocal flops, nbytes
        flops += 4.0 * n * heads * d * dv
        nbytes += (2 if decode else 1) * len(lens) * heads * d * dv * 4
    if case["family"] == "qwen3":
        raw = _qwen3(case)
        W, H, G, vocab = raw["hidden_size"], raw["num_attention_heads"], raw["num_key_value_heads"], raw["vocab_size"]
        for _ in range(raw["num_hidden_layers"]):
            dense((H + 2 * G) * 128, W), dense(W, H * 128), dense(3 * raw["intermediate_size"], W)
            attend(H, 128, 128, G)
    else:
        raw = _config(case)
        W, vocab = raw["width"], VOCAB
        for layer in raw["layers"]:
            m, mlp, kind = layer["mixer"], layer["mlp"], layer["type"]
            a = m.get("left", m)
            if kind == "rglru":
                dense(3 * m["width"], W), dense(2 * m["width"] // m["blocks"], m["width"])
                nbytes += (2 if decode else 1) * len(lens) * m["width"] * 4
            elif kind in ("lightning", "delta", "channel_delta"):
                G = m.get("kv_heads", m["heads"])
                dense((2 * G + 3 * m["heads"]) * 128, W), memory(m["heads"], 128, 128)
            elif "q_rank" in m:
                H, r, dr = m["heads"], m["kv_rank"], m["rot_dim"]
                dense(m["q_rank"] + (0 if "kv_from" in m else r + dr), W), dense(H * (128 + dr), m["q_rank"]), dense(H * 256, r), dense(W, H * 128)
                attend(H, 128 + dr, 128, 0, (m.get("mask") or {}).get("size", 0))
                nbytes += (sum(x for x, _ in spans) + n) * (r + dr) * esize
            else:
                mask = (a.get("mask") or {}).get("size", 0)
                block = case["family"] == "nokipel"
                own = "kv_from" not in a
                gate = W if kind == "parallel" else 0
                dense(a["heads"] * 256 + (2 if own else 0) * a["kv_heads"] * 128 + (a["heads"] * 128 if gate else 0), W)
                attend(a["heads"], 128, 128, a["kv_heads"], 0 if block else mask, mask if block else 0, own)
                if "right" in m:
                    r = m["right"]
                    inner = r["heads"] * r["vdim"]
                    if "state" in r:
                        dense(3 * inner + 2 * r["state"], W), memory(r["heads"], r["vdim"], r["state"])
                    else:
                        dense(5 * inner, W), memory(r["heads"], 128, 128)
            if mlp["kind"] == "dense":
                dense((2 if case["family"] in ("foduzen", "lobidra") else 3) * mlp["ff"], W)
            else:
                experts(mlp["router"]["experts"], mlp["router"]["top"], mlp["expert"]["ff"], W, 2 if case["family"] == "pefazen" else 3)
                if mlp.get("shared"):
                    dense(3 * mlp["shared"]["ff"], W)
    flops += 2.0 * len(lens) * vocab * W
    nbytes += vocab * W * esize + n * (W * esize + 8) + len(lens) * vocab * esize
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # float32: 32-bit sums in another order (measured against 64 bits: 1e-6); bfloat16: what a stack of layers that round every
    # activation to 8 bits of mantissa keeps (measured against 64 bits: 0.011 to 0.019 over the 28 layers of the benchmark model,
    # 0.003 to 0.007 over the 2 to 4 of the others)
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 0.03, "max": 0.5} if case["size"] == "qwen3-0.6b" else {"rel": 0.02, "max": 0.4}


# ---- the same step in 64 bits, in plain torch -----------------------------------------------------------------------------
def _rms(x, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _softplus(z):
    return torch.logaddexp(z, torch.zeros_like(z))


def _turn(x, freq, mag=1.0, halves=False, start=0):
    """x [..., T, heads, d] from position `start` on: the leading 2 len(freq) entries turn in pairs."""
    half = len(freq)
    ang = torch.arange(start, start + x.shape[-3], dtype=F64, device=x.device)[:, None] * torch.tensor(freq, dtype=F64, device=x.device)
    c, s = (mag * torch.cos(ang))[:, None], (mag * torch.sin(ang))[:, None]
    out = x.clone()
    a, b = (slice(0, half), slice(half, 2 * half)) if halves else (slice(0, 2 * half, 2), slice(1, 2 * half, 2))
    out[..., a], out[..., b] = x[..., a] * c - x[..., b] * s, x[..., b] * c + x[..., a] * s
    return out


def _frequencies(rot):
    """(frequencies of the pairs, factor on cos and sin)."""
    dims, base, sc = rot["dims"], rot["base"], rot.get("scaling")
    f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    if sc and "fast" in sc:
        def mark(turns):
            return dims * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
        lo, hi = max(math.floor(mark(sc["fast"])), 0), min(math.ceil(mark(sc["slow"])), dims - 1)
        ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
        return [x / sc["factor"] * r + x * (1.0 - r) for x, r in zip(f, ramp)], 0.1 * math.log(sc["factor"]) + 1.0
    if sc:
        def band(x):
            length = 2.0 * math.pi / x
            if length < sc["original"] / sc["high"]:
                return x
            s = 0.0 if length > sc["original"] / sc["low"] else (sc["original"] / length - sc["low"]) / (sc["high"] - sc["low"])
            return (1.0 - s) * x / sc["factor"] + s * x
        f = [band(x) for x in f]
    return f, 1.0


def _attend(q, k, v, scale, visible, sink=None, cap=0.0):
    """q [B, T, H, d], k [B, S, G, d], v [B, S, G, dv], visible [T, S] -> [B, T, H, dv]; sink: a score without a value per head."""
    out = torch.zeros(*q.shape[:3], v.shape[-1], dtype=F64, device=q.device)
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            g = h // (q.shape[2] // k.shape[2])
            s = q[b, :, h] @ k[b, :, g].T * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            s = s.masked_fill(~visible, -math.inf)
            m = s.amax(1, keepdim=True)
            if sink is not None:
                m = m.clamp(min=float(sink[h]))
            e = torch.exp(s - m)
            den = e.sum(1, keepdim=True) + (torch.exp(sink[h] - m) if sink is not None else 0.0)
            out[b, :, h] = e @ v[b, :, g] / den
    return out


def _visible(T, window=0, chunk=0):
    i = torch.arange(T, device="cuda")
    see = i[None] <= i[:, None]
    if window:
        see = see & (i[None] > i[:, None] - window)
    return see & (i[None] // chunk == i[:, None] // chunk) if chunk else see


def _memory(q, k, v, logs):
    """Linear recurrence S <- a S + k v^T, o = S^T q with per-step log decays: sum over j <= i of exp(L_i - L_j) (q_i . k_j) v_j.
    q, k [B, T, H, d], v [B, T, H, dv], logs [B, T, H]."""
    L, out = logs.cumsum(1), torch.zeros_like(v)
    see = _visible(q.shape[1])
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            w = torch.exp((L[b, :, None, h] - L[b, None, :, h]).masked_fill(~see, -math.inf))
            out[b, :, h] = (q[b, :, h] @ k[b, :, h].T * w) @ v[b, :, h]
    return out


def _conv(u, w):
    """Causal convolution over time, zeros before the first token: u [B, T, C], w [C, taps]."""
    taps = w.shape[1]
    full = torch.nn.functional.pad(u, (0, 0, taps - 1, 0))
    return sum(full[:, j:j + u.shape[1]] * w[:, j] for j in range(taps))


@torch.inference_mode()
def exact(case, seed):
    if case["family"] == "qwen3":
        return {"logits": _exact_qwen3(case, seed)}
    lens, raw = _lens(case), _config(case)
    weights = _Weights(case, seed, raw)
    ids = _tokens(case, seed, VOCAB)
    tokens = torch.zeros(len(lens), max(lens), dtype=torch.long, device="cuda")
    for i, part in enumerate(ids.split(lens)):
        tokens[i, :lens[i]] = part
    x = _Exact(case["family"], raw, weights, tokens, lens).stream()
    last = x[torch.arange(len(lens)), torch.tensor(lens) - 1]
    fam, W = case["family"], raw["width"]
    head = weights("embed" if fam in ("ligidra", "reselorn") else "head", VOCAB, W).to(F64)
    g = weights("final.norm", *(() if fam == "foduzen" else (W,))).to(F64)
    if fam == "pefazen":
        last = last - last.mean(-1, keepdim=True)
    z = _rms(last) * (1.0 + g if fam == "lobidra" else g) @ head.T
    return {"logits": 30.0 * torch.tanh(z / 30.0) if fam == "pefazen" else z}


class _Exact:
    """Forward of a registry family on padded sequences [B, T] (what follows a sequence's end reaches nothing before it)."""

    def __init__(self, family, raw, weights, tokens, lens):
        self.family, self.raw, self.weights, self.tokens, self.W = family, raw, weights, tokens, raw["width"]
        self.live = torch.arange(tokens.shape[1], device="cuda")[None] < torch.tensor(lens, device="cuda")[:, None]
        self.B, self.T = tokens.shape
        self.kept, self.first = {}, None

    def w(self, name, *shape):
        return self.weights(name, *shape).to(F64) if name.split(".")[-1] != "table" else self.weights(name, *shape)

    def lin(self, x, name, out, width=None):
        return x @ self.w(name, out, width or self.W).T

    def heads(self, x, h):
        return x.view(self.B, self.T, h, -1)

    def stream(self):
        W, fam = self.W, self.family
        e = self.w("embed", VOCAB, W)
        x = e[self.tokens]
        if fam == "foduzen":
            ang = torch.arange(self.T, dtype=F64, device="cuda")[:, None] * torch.pow(10000.0, -2.0 * torch.arange(W // 2, dtype=F64, device="cuda") / W)
            x = x + torch.stack([torch.sin(ang), torch.cos(ang)], -1).view(self.T, W)
        if fam == "ligidra":
            x = _rms(x) * self.w("embed.norm", W)
            side = self.w("side.embed", VOCAB, len(self.raw["layers"]) * W // 16)[self.tokens]
        for i, layer in enumerate(self.raw["layers"]):
            p = f"l{layer.get('weights_of', i)}."
            mix = getattr(self, "mix_" + fam)
            if fam == "foduzen":
                x = x + _rms(mix(x, p + "mix.", layer)) * self.w(p + "norm1")
                u = self.w(p + "mlp.act", 2)
                z = self.lin(x, p + "mlp.up", 3 * W)
                zn = z.clamp(max=0.0)
                z = torch.where(z > 0, _softplus(u[0]) * z * z, (0.5 + _softplus(u[1])) * (torch.expm1(zn) - zn)) + 0.5 * z
                x = x + _rms(self.lin(z, p + "mlp.down", W, 3 * W)) * self.w(p + "norm2")
            elif fam == "nokipel":
                x = x + mix(_rms(x) * self.w(p + "norm1", W), p + "mix.", layer)
                h = _rms(x) * self.w(p + "norm2", W)
                x = x + (self.routed(h, p + "mlp.", layer["mlp"]) if layer["mlp"]["kind"] == "moe" else self.clamped(h, p + "mlp."))
            elif fam == "pefazen":
                h = x - x.mean(-1, keepdim=True)
                x = x + mix(_rms(h) * self.w(p + "norm1", W), i, layer)
                h = x - x.mean(-1, keepdim=True)
                x = x + self.routed(_rms(h) * self.w(p + "norm2", W), p + "mlp.", layer["mlp"])
            elif fam == "lobidra":
                y = mix(_rms(x) * (1.0 + self.w(p + "norm1", W)), p + "mix.", layer)
                x = x + _rms(y) * (1.0 + self.w(p + "norm1b", W))
                h = _rms(x) * (1.0 + self.w(p + "norm2", W))
                y = self.routed(h, p + "mlp.", layer["mlp"]) if layer["mlp"]["kind"] == "moe" else \
                    self.lin(_gelu(self.lin(h, p + "mlp.up", 3 * W)), p + "mlp.down", W, 3 * W)
                x = x + _rms(y) * (1.0 + self.w(p + "norm2b", W))
            elif fam == "ligidra":
                h = _rms(x) * self.w(p + "norm1", W)
                before = torch.nn.functional.pad(h, (0, 0, 1, 0))[:, :-1]
                x = x + mix(h + (before - h) * self.w(p + "shift", W), i, layer)
                x = x + self.routed(_rms(x) * self.w(p + "norm2", W), p + "mlp.", layer["mlp"])
                n = W // 16
                y = self.lin(_gelu(self.lin(x, p + "side.gate", n)) * side[..., i * n:(i + 1) * n], p + "side.proj", W, n)
                x = x + _rms(y) * self.w(p + "side.norm", W)
            else:
                x = x + _rms(mix(x, p + "mix.", layer)) * self.w(p + "norm1", W) * self.w(p + "ls1", W)
                y = self.routed(x, p + "mlp.", layer["mlp"]) if layer["mlp"]["kind"] == "moe" else self.glu(x, p + "mlp.", 3 * W)
                x = x + _rms(y) * self.w(p + "norm2", W) * self.w(p + "ls2", W)
        return x

    # -- mixers
    def mix_foduzen(self, x, p, layer):
        m, W, B, T = layer["mixer"], self.W, self.B, self.T
        if layer["type"] == "rglru":
            C, nb = m["width"], m["blocks"]
            y = _gelu(self.lin(x, p + "y", C) + self.w(p + "y.b", C))
            u = _conv(self.lin(x, p + "x", C) + self.w(p + "x.b", C), self.w(p + "conv", C, 4)) + self.w(p + "conv.b", C)
            bw = C // nb
            ub = u.view(B, T, nb, bw)

            def gate(name):
                w, b = self.w(p + name, nb, bw, bw), self.w(p + name + ".b", nb, bw)
                return torch.sigmoid(torch.stack([ub[:, :, j] @ w[j].T + b[j] for j in range(nb)], 2)).view(B, T, C)
            a = torch.exp(-8.0 * gate("ra") * _softplus(self.w(p + "lam", C)))
            put, S = torch.sqrt(1.0 - a * a) * gate("ri") * u, torch.zeros(B, C, dtype=F64, device="cuda")
            out = torch.empty_like(u)
            for t in range(T):
                S = a[:, t] * S + put[:, t]
                out[:, t] = S
            return self.lin(out * y, p + "o", W, C)
        a, r = m["left"], m["right"]
        H, G = a["heads"], a["kv_heads"]

        def biased(name, n):
            return self.lin(x, p + name, n) + self.w(p + name + ".b", n)
        q = _rms(self.heads(biased("left.q", H * 128), H)) * self.w(p + "left.q.norm", 128)
        k = _rms(self.heads(biased("left.k", G * 128), G)) * self.w(p + "left.k.norm", 128)
        o = _attend(q, k, self.heads(biased("left.v", G * 128), G), a["scale"], _visible(T, window=1024)).view(B, T, -1)
        left = self.lin(o * torch.sigmoid(self.lin(x, p + "left.g", H * 128)), p + "left.o", W, H * 128) + self.w(p + "left.o.b", W)
        Hn, P, N = r["heads"], r["vdim"], r["state"]
        inner, ch = Hn * P, Hn * P + 2 * N
        z, xbc, dt = self.lin(x, p + "right.in", inner + ch + Hn).split([inner, ch, Hn], -1)
        xbc = _silu(_conv(xbc, self.w(p + "right.conv", ch, 4)) + self.w(p + "right.conv.b", ch))
        xs, Bm, Cm = xbc.split([inner, N, N], -1)
        xs, dt = self.heads(xs, Hn), _softplus(dt + self.w(p + "right.dt_bias", Hn))
        wide = (B, T, Hn, N)
        y = _memory(Cm[:, :, None].expand(wide), Bm[:, :, None].expand(wide), xs * dt[..., None], -torch.exp(self.w(p + "right.A_log", Hn)) * dt)
        y = (y + self.w(p + "right.D", Hn)[:, None] * xs).reshape(B, T, inner) * _silu(z)
        right = self.lin(_rms(y) * self.w(p + "right.norm", inner), p + "right.o", W, inner)
        return 0.5 * (_rms(left) * self.w(p + "left.out", W) + _rms(right) * self.w(p + "right.out", W))

    def mix_nokipel(self, h, p, layer):
        m, W, B, T = layer["mixer"], self.W, self.B, self.T
        H = m["heads"]
        if layer["type"] == "lightning":
            q, k, v = (self.heads(_silu(self.lin(h, p + c, H * 128)), H) for c in "qkv")
            logs = torch.tensor(m["decay"], dtype=F64, device="cuda").log().expand(B, T, H)
            y = _rms(_memory(q, k, v, logs).reshape(B, T, -1)) * self.w(p + "norm", H * 128)
            return self.lin(y * torch.sigmoid(self.lin(h, p + "g", H * 128)), p + "o", W, H * 128)
        f, _ = _frequencies(m["rot"])
        q, k, v = (self.heads(self.lin(h, p + c, n * 128) + self.w(p + c + ".b", n * 128), n) for c, n in (("q", H), ("k", m["kv_heads"]), ("v", m["kv_heads"])))
        o = _attend(_turn(q, f), _turn(k, f), v, m["scale"], _visible(T, chunk=1024))
        return self.lin(o.view(B, T, -1), p + "o", W, H * 128)

    def mix_pefazen(self, h, i, layer):
        m, p, W, B, T = layer["mixer"], f"l{i}.mix.", self.W, self.B, self.T
        H, r, dr, qr, second = m["heads"], m["kv_rank"], m["rot_dim"], m["q_rank"], layer["type"].endswith("2")
        f, mag = _frequencies(m["rot"])
        if "kv_from" in m:
            lat, kr = self.kept[m["kv_from"]]
        else:
            down = self.lin(h, p + "dkv", r + dr)
            lat, kr = _rms(down[..., :r]) * self.w(p + "dkv.norm", r), _turn(down[..., None, r:], f, mag, second)
            self.kept[i] = lat, kr
        q = self.heads(self.lin(_rms(self.lin(h, p + "dq", qr)) * self.w(p + "dq.norm", qr), p + "uq", H * (128 + dr), qr), H)
        q = torch.cat([q[..., :128], _turn(q[..., 128:], f, mag, second)], -1)
        k = torch.cat([self.heads(self.lin(lat, p + "uk", H * 128, r), H), kr.expand(B, T, H, dr)], -1)
        o = _attend(q, k, self.heads(self.lin(lat, p + "uv", H * 128, r), H), m["scale"], _visible(T, window=0 if second else 1024))
        if not second:
            o = o * torch.sigmoid(self.lin(h, p + "g", H))[..., None]
        return self.lin(o.view(B, T, -1), p + "o", W, H * 128)

    def mix_lobidra(self, h, p, layer):
        m, W, B, T = layer["mixer"], self.W, self.B, self.T
        if layer["type"] == "attention":
            H, G = m["heads"], m["kv_heads"]
            f, _ = _frequencies(m["rot"])
            q = self.heads(_conv(self.lin(h, p + "q", H * 128), self.w(p + "q.conv", H * 128, 4)), H)
            k = self.heads(_conv(self.lin(h, p + "k", G * 128), self.w(p + "k.conv", G * 128, 4)), G)
            o = _attend(_turn(q, f), _turn(k, f), k, m["scale"], _visible(T), torch.zeros(H, dtype=F64, device="cuda"))
            o = o * torch.sigmoid(self.lin(h, p + "g", H))[..., None]
            return self.lin(o.view(B, T, -1), p + "o", W, H * 128)
        a, r, pl, pr = m["left"], m["right"], p + "left.", p + "right."
        H, G = a["heads"], a["kv_heads"]
        at = torch.arange(T, dtype=F64, device="cuda")
        temp = 1.0 + a["q_temp"]["coef"] * torch.log(torch.floor((at + 1.0) / a["q_temp"]["every"]) + 1.0)
        q, k, v = (self.heads(self.lin(h, pl + c, n * 128), n) for c, n in (("q", H), ("k", G), ("v", G)))
        o = _attend(q * temp[:, None, None], k, v, a["scale"], _visible(T), self.w(pl + "sink", H)).view(B, T, -1)
        left = self.lin(o * torch.sigmoid(self.lin(h, pl + "g", H * 128)), pl + "o", W, H * 128)
        H, cap = r["heads"], r["gate_cap"]
        q, k, v = (self.heads(self.lin(h, pr + c, H * 128), H) for c in "qkv")
        gi = cap * torch.tanh((self.lin(h, pr + "i", H) + self.w(pr + "i.b", H)) / cap)
        F = -_softplus(-cap * torch.tanh((self.lin(h, pr + "f", H) + self.w(pr + "f.b", H)) / cap))
        F = F.cumsum(1)
        mx = F + (gi - F).cummax(1)[0].clamp(min=0.0)        # the running maximum, 0 before the first token
        out, see = torch.zeros_like(v), _visible(T)
        for b in range(B):
            for j in range(H):
                wt = torch.exp((F[b, :, None, j] - F[b, None, :, j] + gi[b, None, :, j] - mx[b, :, None, j]).masked_fill(~see, -math.inf))
                wt = wt * (q[b, :, j] @ k[b, :, j].T) * 128 ** -0.5
                out[b, :, j] = wt @ v[b, :, j] / (torch.maximum(wt.sum(1).abs(), torch.exp(-mx[b, :, j])) + 1e-6)[:, None]
        y = _rms(out).reshape(B, T, -1) * self.w(pr + "norm", H * 128) * torch.sigmoid(self.lin(h, pr + "g", H * 128))
        return m["left_scale"] * left + m["right_scale"] * self.lin(y, pr + "o", W, H * 128)

    def mix_ligidra(self, h, i, layer):
        m, p, W, B, T = layer["mixer"], f"l{i}.mix.", self.W, self.B, self.T
        H, G = m["heads"], m["kv_heads"]
        if layer["type"] == "attention":
            f, _ = _frequencies(m["rot"])
            q = _turn(self.heads(_rms(self.lin(h, p + "q", H * 128)) * self.w(p + "q.norm", H * 128), H), f)
            if "kv_from" not in m:
                k = _turn(self.heads(_rms(self.lin(h, p + "k", G * 128)) * self.w(p + "k.norm", G * 128), G), f)
                self.kept[i] = k, self.heads(self.lin(h, p + "v", G * 128), G)
            k, v = self.kept[m.get("kv_from", i)]
            size, pool = m["mask"]["size"], m["mask"]["pool"]
            nb = T // pool
            means = [x[:, :nb * pool].reshape(B, nb, pool, G, 128).mean(2) for x in (k, v)]
            end = torch.arange(nb, device="cuda") * pool + pool - 1
            see = torch.cat([_visible(T, window=size), end[None] <= torch.arange(T, device="cuda")[:, None] - size], 1)
            o = _attend(q, torch.cat([k, means[0]], 1), torch.cat([v, means[1]], 1), m["scale"], see, self.w(p + "sink", H), m["softcap"])
            return self.lin(o.view(B, T, -1), p + "o", W, H * 128)

        def conv(c, n):
            return self.heads(_silu(_conv(self.lin(h, p + c, n * 128), self.w(p + c + ".conv", n * 128, 4))), n)

        def unit(x):
            return (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 2)
        q, k, v = unit(conv("q", G)) * 128 ** -0.5, unit(conv("k", G)), conv("v", H)
        beta, rate = torch.sigmoid(self.lin(h, p + "b", H)), torch.exp(self.w(p + "A_log", H))
        if layer["type"] == "channel_delta":
            z = self.lin(self.lin(h, p + "a1", 128), p + "a2", H * 128, 128) + self.w(p + "dt_bias", H * 128)
            decay = torch.exp(-rate[:, None] * _softplus(self.heads(z, H)))
            gate = torch.sigmoid(self.lin(self.lin(h, p + "g1", 128), p + "g2", H * 128, 128))
        else:
            decay = torch.exp(-rate * _softplus(self.lin(h, p + "a", H) + self.w(p + "dt_bias", H)))[..., None]
            gate = _silu(self.lin(h, p + "g", H * 128))
        S, o = torch.zeros(B, H, 128, 128, dtype=F64, device="cuda"), torch.empty_like(v)
        for t in range(T):
            S = S * decay[:, t, :, :, None]
            u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None] @ S)[:, :, 0])
            S = torch.addcmul(S, k[:, t, :, :, None], u[:, :, None])
            o[:, t] = (q[:, t, :, None] @ S)[:, :, 0]
        return self.lin((_rms(o) * self.w(p + "norm", 128)).view(B, T, -1) * gate, p + "o", W, H * 128)

    def mix_reselorn(self, x, p, layer):
        m, W, B, T = layer["mixer"], self.W, self.B, self.T
        H, G = m["heads"], m["kv_heads"]
        f, mag = _frequencies(m["rot"])
        q, k, v = (self.heads(self.lin(x, p + c, n * 128), n) for c, n in (("q", H), ("k", G), ("v", G)))
        q, k = _rms(_turn(q, f, mag, True)), _rms(_turn(k, f, mag, True))
        if self.first is None:
            self.first = v
        else:
            lam = self.w(p + "vmix")
            v = (1.0 - lam) * v + lam * self.first
        o = _attend(q, k, v, m["scale"], _visible(T, window=1024), self.w(p + "sink", H))
        return self.lin(o.view(B, T, -1), p + "o", W, H * 128)

    # -- feed-forwards
    def glu(self, h, p, ff):
        return self.lin(_silu(self.lin(h, p + "gate", ff)) * self.lin(h, p + "up", ff), p + "down", self.W, ff)

    def clamped(self, h, p):
        ff = 3 * self.W
        g, u = self.lin(h, p + "gate", ff).clamp(max=7.0), self.lin(h, p + "up", ff).clamp(-7.0, 7.0)
        return self.lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "down", self.W, ff)

    def routed(self, h, p, mlp):
        r, fam, W, ff = mlp["router"], self.family, self.W, mlp["expert"]["ff"]
        E, top, total = r["experts"], r["top"], r["experts"] + r.get("identity", 0)
        flat, live = h.reshape(-1, W), self.live.view(-1)
        z = flat @ self.w(p + "router", total, W).T if fam != "lobidra" else None
        if fam == "lobidra":
            idx = self.w(p + "table", VOCAB, top)[self.tokens.view(-1)].long()
            wt = torch.full(idx.shape, 1.0 / top, dtype=F64, device="cuda")
        elif fam == "reselorn":
            val, idx = (z + self.w(p + "router.b", total)).topk(top, 1)
            wt = torch.softmax(val, 1)
        elif fam == "ligidra":
            wt, idx = torch.softmax(z, 1).topk(top, 1)
        elif fam == "pefazen":
            s = torch.sigmoid(z)
            idx = (s + self.w(p + "correction", total)).topk(top, 1)[1]
            wt = s.gather(1, idx)
        else:
            s, g = torch.softmax(z, 1), r["groups"]
            c = (s + self.w(p + "correction", total)).view(-1, g["count"], total // g["count"])
            kept = c.amax(2).topk(g["keep"], 1)[1]
            c = c.masked_fill(torch.ones_like(c[..., 0], dtype=torch.bool).scatter(1, kept, False)[..., None], -math.inf).view(-1, total)
            idx = c.topk(top, 1)[1]
            wt = s.gather(1, idx)
            wt = wt / (wt.sum(1, keepdim=True) + 1e-20) * r["scale"]
        out = torch.zeros_like(flat)
        for e in range(total):
            row, place = torch.nonzero((idx == e) & live[:, None], as_tuple=True)
            if not row.numel():
                continue
            a, q = flat[row], f"{p}e{e}."
            if e >= E:
                y = a
            elif fam == "pefazen":
                y = self.lin(self.lin(a, q + "up", ff).clamp(min=0.0) ** 2, q + "down", W, ff)
            else:
                y = self.glu(a, q, ff)
            out.index_add_(0, row, y * wt[row, place][:, None])
        out = out.view(h.shape)
        if mlp.get("shared"):
            y = self.glu(h, p + "shared.", mlp["shared"]["ff"])
            out = out + (y * torch.sigmoid(self.lin(h, p + "shared.sg", 1)) if fam == "nokipel" else y)
        return out


def _exact_qwen3(case, seed):
    raw, lens, cached, decode = _qwen3(case), _lens(case), case["cached"], case["step"] == "decode"
    W, H, G, ff, vocab = raw["hidden_size"], raw["num_attention_heads"], raw["num_key_value_heads"], raw["intermediate_size"], raw["vocab_size"]
    get = _Weights(case, seed, raw)

    def w(name, *shape):
        return get(name, *shape).to(F64)
    table, pages = _page_table([n + cached for n in lens], seed)
    ids = _tokens(case, seed, vocab)
    ids = ids[torch.tensor(lens).cumsum(0).sub(1).cuda()] if decode else ids
    spans = [(n - 1, n) if decode else (cached, cached + n) for n in lens]
    at = torch.tensor([0] + [b - a for a, b in spans]).cumsum(0).tolist()
    f, _ = _frequencies({"dims": 128, "base": raw["rope_theta"]})

    def turn(x):                                             # packed rows, each sequence from its own position on
        return torch.cat([_turn(x[s:e], f, halves=True, start=a) for (a, _), s, e in zip(spans, at, at[1:])])
    x = w("model.embed_tokens.weight", vocab, W)[ids]
    for i in range(raw["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = _rms(x) * w(p + "input_layernorm.weight", W)
        q = (h @ w(p + "self_attn.q_proj.weight", H * 128, W).T).view(-1, H, 128)
        k = (h @ w(p + "self_attn.k_proj.weight", G * 128, W).T).view(-1, G, 128)
        v = (h @ w(p + "self_attn.v_proj.weight", G * 128, W).T).view(-1, G, 128)
        q = turn(_rms(q) * w(p + "self_attn.q_norm.weight", 128))
        k = turn(_rms(k) * w(p + "self_attn.k_norm.weight", 128))
        o = torch.empty_like(q)
        kv = _cached_kv(case, seed, i, pages, G) if decode or cached else None
        for j, ((a, b), s, e) in enumerate(zip(spans, at, at[1:])):
            ks, vs = k[s:e], v[s:e]
            if a:
                rows = table[j, :-(-a // PAGE)].long().cuda()
                ks, vs = (torch.cat([c[rows].transpose(1, 2).reshape(-1, G, 128)[:a].to(F64), new]) for c, new in zip(kv, (ks, vs)))
            see = torch.arange(b, device="cuda")[None] <= torch.arange(a, b, device="cuda")[:, None]
            if decode:
                sc = torch.einsum("ghd,sgd->ghs", q[s].view(G, H // G, 128), ks) * 128 ** -0.5
                o[s] = torch.einsum("ghs,sgd->ghd", torch.softmax(sc, -1), vs).reshape(H, 128)
            else:
                o[s:e] = _attend(q[None, s:e], ks[None], vs[None], 128 ** -0.5, see)[0]
        x = x + o.view(-1, H * 128) @ w(p + "self_attn.o_proj.weight", W, H * 128).T
        h = _rms(x) * w(p + "post_attention_layernorm.weight", W)
        h = _silu(h @ w(p + "mlp.gate_proj.weight", ff, W).T) * (h @ w(p + "mlp.up_proj.weight", ff, W).T)
        x = x + h @ w(p + "mlp.down_proj.weight", W, ff).T
    x = x[torch.tensor(at[1:]).sub(1).cuda()]
    head = w("model.embed_tokens.weight" if raw["tie_word_embeddings"] else "lm_head.weight", vocab, W)
    return _rms(x) * w("model.norm.weight", W) @ head.T
