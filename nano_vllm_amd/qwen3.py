"""Qwen3 decoder built on the libnvl kernels — the only model family the reference ships
(nano-vllm models/qwen3.py:14-216). Same module tree and parameter names as the reference /
HF checkpoints (so `packed_modules_mapping`-style loading works), but the per-layer dataflow
is arranged for MI355X:

   add+RMSNorm -> qkv GEMM -> [q/k-norm + RoPE + KV-cache store: ONE launch]
               -> paged decode attention | MFMA prefill attention -> o GEMM (+all-reduce)
   add+RMSNorm -> gate_up GEMM -> SiLU*mul -> down GEMM (+all-reduce)

i.e. 10 launches per layer instead of the reference's 13 (each dependent kernel boundary is
~1.5 us on this chip even inside a hipGraph; a small dependent
kernel costs ~5 us whatever it does). On decode-sized batches (<= 256 rows, TP=1, single-K-pass
shapes) the chain is 8 launches:

   add+RMSNorm(fp32 slabs) -> qkv GEMM -> [q/k-norm + RoPE + KV store + paged attention: ONE launch]
   -> split merge -> o GEMM (fp32 split-K slabs) -> add+RMSNorm(slabs) -> gate_up GEMM + SiLU*mul epilogue
   -> down GEMM (slabs)

with the GEMMs on the hand-written skinny kernel (nvl_linear_decode). Up to 8 rows (TP=1, width <= 1024) it is 5 or 6 (up to 4 rows the o GEMM merges
the parts of a context, beyond them a launch of its own):

   [add+RMSNorm + qkv GEMM] -> [norm + RoPE + KV store + attention, split merged in LDS] -> o GEMM
   -> [add+RMSNorm + gate_up GEMM + SiLU*mul] -> down GEMM

and up to 4 rows of Qwen3-0.6B's shape all layers are one launch (decode_step.hip).
"""
from __future__ import annotations

import os

import torch
from torch import nn
from torch.nn.modules import module as _hooks

from .api import model_geometry
from .attn_meta import get_context, plain_calls
from .layers import (Attention, MergedColumnParallelLinear, ParallelLMHead, QKVParallelLinear, RMSNorm,
                     RowParallelLinear, SiluAndMul, VocabParallelEmbedding, get_rope)
from . import ops, ops_seq, tp


class Qwen3Attention(nn.Module):

    def __init__(self, geo: dict, total_heads: int, total_kv_heads: int, qkv_bias: bool):
        super().__init__()
        self.num_heads, self.num_kv_heads, self.head_dim = geo["heads"], geo["kv_heads"], geo["head_dim"]
        self.q_size = self.num_heads * self.head_dim
        self.kv_size = self.num_kv_heads * self.head_dim
        self.eps = geo["eps"]
        self.qkv_proj = QKVParallelLinear(geo["hidden"], self.head_dim, total_heads, total_kv_heads, bias=qkv_bias)
        self.o_proj = RowParallelLinear(total_heads * self.head_dim, geo["hidden"], bias=False)
        self.rotary_emb = get_rope(self.head_dim, self.head_dim, geo["max_pos"], geo["rope_theta"])
        self.attn = Attention(self.num_heads, self.head_dim, self.head_dim ** -0.5, self.num_kv_heads)
        self.has_qk_norm = not qkv_bias                      # models/qwen3.py:68-70
        if self.has_qk_norm:
            self.q_norm = RMSNorm(self.head_dim, eps=self.eps)
            self.k_norm = RMSNorm(self.head_dim, eps=self.eps)

    def forward(self, positions: torch.Tensor, hidden_states: torch.Tensor, qkv: torch.Tensor | None = None) -> torch.Tensor:
        """qkv: the projection of hidden_states, where the norm in front of it has made it already."""
        ctx = get_context()
        # (a step whose plan carries a shared prefix takes bf16 qkv: the attention kernel that also serves the shared-prefix packs
        #  in the SAME launch has no scalar registers left for the slab-sum prologue — attn_decode.hip — and with slabs the pass
        #  would be a launch of its own on a divided grid)
        if qkv is not None:
            pass
        elif self.attn.fuses_decode_step(ctx) and not ctx.shared_prefix:
            qkv = self.qkv_proj.forward_for_fused_decode(hidden_states)      # bf16 [N, out], or fp32 split-K slabs
        else:
            qkv = self.qkv_proj(hidden_states)
        qw = self.q_norm.weight if self.has_qk_norm else None
        kw = self.k_norm.weight if self.has_qk_norm else None
        if not ctx.is_prefill:
            y = self.attn.forward_open(qkv, qw, kw, self.eps, self.rotary_emb.cos_sin_cache, self.o_proj)
            if y is not None:
                return y
        o = self.attn.forward_fused(qkv, positions, qw, kw, self.eps, self.rotary_emb.cos_sin_cache)
        return self.o_proj.forward_decode(o.view(o.shape[0], -1))


class Qwen3MLP(nn.Module):

    def __init__(self, hidden_size: int, intermediate_size: int, hidden_act: str):
        super().__init__()
        assert hidden_act == "silu"
        self.gate_up_proj = MergedColumnParallelLinear(hidden_size, [intermediate_size] * 2, bias=False)
        self.down_proj = RowParallelLinear(intermediate_size, hidden_size, bias=False)
        self.act_fn = SiluAndMul()

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.down_proj.forward_decode(self.gate_up_proj.forward_silu(x))

    def forward_normed(self, norm: RMSNorm, x, residual):
        """(self(norm(x, residual)), the new residual) of a decode step; few rows take norm, gate|up and activation in one launch."""
        both = norm.into_linear(x, residual, self.gate_up_proj, silu=True)
        if both is not None:
            return self.down_proj.forward_decode(both[0]), both[1]
        hidden_states, residual = norm(x, residual)
        return self(hidden_states), residual


def _watched(*modules) -> bool:
    """Does anybody look at these modules' calls? Then they are called, with their own inputs and outputs."""
    return bool(_hooks._global_forward_hooks or _hooks._global_forward_pre_hooks or any(m._forward_hooks or m._forward_pre_hooks for m in modules))


class Qwen3DecoderLayer(nn.Module):

    def __init__(self, config, geo: dict):
        super().__init__()
        self.self_attn = Qwen3Attention(geo, config.num_attention_heads, config.num_key_value_heads,
                                        qkv_bias=getattr(config, "attention_bias", True))     # default as models/qwen3.py:133
        self.mlp = Qwen3MLP(config.hidden_size, config.intermediate_size, config.hidden_act)
        self.input_layernorm = RMSNorm(config.hidden_size, eps=config.rms_norm_eps)
        self.post_attention_layernorm = RMSNorm(config.hidden_size, eps=config.rms_norm_eps)

    def forward(self, positions, hidden_states, residual):
        attn, qkv = self.self_attn, None
        decode = attn.qkv_proj.tp_size == 1 and not get_context().is_prefill
        if decode and not _watched(self.input_layernorm, attn):
            both = self.input_layernorm.into_linear(hidden_states, residual, attn.qkv_proj)
            if both is not None:
                qkv, residual = both
        if qkv is None:
            if residual is None:                             # first layer: residual = embeddings
                residual = hidden_states
                hidden_states = self.input_layernorm(hidden_states)
            else:
                hidden_states, residual = self.input_layernorm(hidden_states, residual)
        hidden_states = attn(positions, hidden_states) if qkv is None else attn(positions, hidden_states, qkv)
        if decode and not _watched(self.post_attention_layernorm, self.mlp):
            return self.mlp.forward_normed(self.post_attention_layernorm, hidden_states, residual)
        hidden_states, residual = self.post_attention_layernorm(hidden_states, residual)
        return self.mlp(hidden_states), residual


# The calls of a decode step that ops.decode_step stands in for, by class, and what they are as the files have them
_CALLS = {Qwen3DecoderLayer: {"forward"}, Qwen3Attention: {"forward"}, Qwen3MLP: {"forward", "forward_normed"}, RMSNorm: {"forward", "into_linear"},
          Attention: {"forward_open", "forward_fused", "fuses_decode_step"}, QKVParallelLinear: {"forward", "forward_for_fused_decode"},
          RowParallelLinear: {"forward", "forward_decode"}, MergedColumnParallelLinear: {"forward", "forward_silu"}}
_OWN = {kind: frozenset(names | {"weight", "bias"}) for kind, names in _CALLS.items()}        # what an instance may not have of its own
_AS_MADE = [(kind, name, getattr(kind, name)) for kind, names in _CALLS.items() for name in (*names, "__call__")]


def _as_made() -> bool:
    """Has nobody replaced one of these calls in its class, or watches all modules?"""
    return not (_hooks._global_forward_hooks or _hooks._global_forward_pre_hooks) and all(getattr(kind, name) is call for kind, name, call in _AS_MADE)


def _plain(module, kind) -> bool:
    """Is the module of that class itself, with no call of its own and nobody watching? (of a class that is as made)"""
    return type(module) is kind and module.__dict__.keys().isdisjoint(_OWN[kind]) and not module._forward_hooks and not module._forward_pre_hooks


def _step_layer(layer):
    """What ops.decode_step takes of a layer: what all layers have in common (eps, heads, kv heads, scale, matrices' and caches' shapes; the rotary table) and its own tensors. None: a
    layer that is not as this file makes it; nothing is read of a module before it is known to be."""
    if not _plain(layer, Qwen3DecoderLayer):
        return None
    m = layer._modules                           # (a module's attributes go through Python otherwise: 680 us a step of 28 layers, 430 so)
    attn, mlp, n1, n2 = m.get("self_attn"), m.get("mlp"), m.get("input_layernorm"), m.get("post_attention_layernorm")
    if not (_plain(attn, Qwen3Attention) and _plain(mlp, Qwen3MLP) and _plain(n1, RMSNorm) and _plain(n2, RMSNorm)):
        return None
    m, f = attn._modules, mlp._modules
    a, qkv, o, gate_up, down = m.get("attn"), m.get("qkv_proj"), m.get("o_proj"), f.get("gate_up_proj"), f.get("down_proj")
    if not (_plain(a, Attention) and _plain(qkv, QKVParallelLinear) and _plain(o, RowParallelLinear) and _plain(gate_up, MergedColumnParallelLinear)
            and _plain(down, RowParallelLinear) and qkv.tp_size == 1):
        return None
    if any(p._parameters.get("bias", 0) is not None for p in (qkv, o, gate_up, down)):        # (0: it is kept elsewhere)
        return None
    eps, table, normed = n1.eps, attn.rotary_emb.cos_sin_cache, attn.has_qk_norm
    if n2.eps != eps or a.num_heads != attn.num_heads or a.num_kv_heads != attn.num_kv_heads or a.k_cache.numel() == 0 or normed and attn.eps != eps:
        return None
    w = [p._parameters.get("weight") for p in (n1, qkv, o, n2, gate_up, down)]
    if any(t is None for t in w):
        return None
    tensors = (w[0], w[1], attn.q_norm.weight if normed else None, attn.k_norm.weight if normed else None, *w[2:], a.k_cache, a.v_cache)
    at = 0
    for t in tensors:
        if t is not None:
            if t.dtype != torch.bfloat16 or not t.is_contiguous():
                return None
            at |= t.data_ptr()
    common = (eps, attn.num_heads, attn.num_kv_heads, a.scale, w[1].shape, w[2].shape, w[4].shape, w[5].shape, a.k_cache.shape, a.v_cache.shape)
    return None if at % 16 else (common, table, tensors)


# NVL_DECODE_STEP=0 keeps the launches of small decode steps apart (A/B measurements)
_DECODE_STEP = os.environ.get("NVL_DECODE_STEP", "1") != "0"
# The longest context (max_context) up to which that many sequences' layers go in one launch: its attention has 30, 28, 24 and 24 parts for each
# pair of heads, and the launches of their own use the whole chip. Qwen3-0.6B, us a step, apart / in one: one sequence of 8,000, 16,000, 30,000 tokens 970 1144 1414 / 727 894 1216;
# two of 8,000 1111 / 920; three of 4,000 1007 / 907, of 8,000 1255 / 1257; four of 4,000 1094 / 1035, of 8,000 1379 / 1475. Shorter contexts: decode_step.hip.
_DECODE_STEP_CONTEXT = {1: 32768, 2: 8192, 3: 4096, 4: 4096}


class Qwen3Model(nn.Module):

    def __init__(self, config, geo: dict):
        super().__init__()
        self.embed_tokens = VocabParallelEmbedding(config.vocab_size, config.hidden_size)
        self.layers = nn.ModuleList([Qwen3DecoderLayer(config, geo) for _ in range(config.num_hidden_layers)])
        self.norm = RMSNorm(config.hidden_size, eps=config.rms_norm_eps)

    def _decode_step(self, x: torch.Tensor):
        """All layers of a decode step of few sequences in one launch (decode_step.hip): (the last layer's output, the residual), or None where the layers are called: other
        steps and shapes, and layers of which somebody watches, replaces or extends a part."""
        ctx = get_context()
        if (not _DECODE_STEP or ctx.is_prefill or x.dim() != 2 or not 1 <= x.shape[0] <= ops.DECODE_STEP_MAX_ROWS or x.dtype != torch.bfloat16 or not x.is_cuda
                or not x.is_contiguous() or ctx.shared_prefix or ctx.context_lens is None or ctx.block_tables is None or not len(self.layers)):
            return None
        first = _step_layer(self.layers[0]) if _as_made() else None
        if first is None:
            return None
        common, table, tensors = first
        eps, hq, hkv, scale, *shapes, cache, _ = common
        W, ff = x.shape[1], shapes[3][-1]
        if (not self.layers[0].self_attn.attn.fuses_decode_step(ctx) or not ops.decode_step_bytes(x.shape[0], len(self.layers), W, ff, hq, hkv)
                or shapes != [((hq + 2 * hkv) * 128, W), (W, hq * 128), (2 * ff, W), (W, ff)] or len(cache) != 4 or cache != common[-1]):
            return None
        tables, block_size, ws = ctx.block_tables, cache[2], ctx.decode_workspace
        max_context = ctx.max_context or tables.shape[1] * block_size
        if (max_context > _DECODE_STEP_CONTEXT[x.shape[0]] or block_size % 32 or tables.stride(0) * block_size < max_context or tables.stride(1) != 1
                or ws is not None and ws.numel() * ws.element_size() < ops.paged_attn_decode_workspace_bytes(x.shape[0], hq, max_context)):
            return None                          # (what the layers' own launches refuse they still do)
        layers = [tensors]
        for layer in list(self.layers)[1:]:
            other = _step_layer(layer)
            if other is None or other[0] != common or other[1] is not table:
                return None
            layers.append(other[2])
        return ops.decode_step(x, layers, eps, table, tables, ctx.context_lens, ff, hq, scale, gave_up=ctx.decode_gave_up)

    def forward(self, input_ids: torch.Tensor, positions: torch.Tensor) -> torch.Tensor:
        hidden_states = self.embed_tokens(input_ids)
        residual = None
        both = self._decode_step(hidden_states)
        if both is not None:
            hidden_states, residual = both
        else:
            for layer in self.layers:
                hidden_states, residual = layer(positions, hidden_states, residual)
        hidden_states, _ = self.norm(hidden_states, residual)
        return hidden_states


class Qwen3ForCausalLM(nn.Module):
    # checkpoint-name fragment -> (fused parameter fragment, shard id)   (models/qwen3.py:187-193)
    packed_modules_mapping = {
        "q_proj": ("qkv_proj", "q"),
        "k_proj": ("qkv_proj", "k"),
        "v_proj": ("qkv_proj", "v"),
        "gate_proj": ("gate_up_proj", 0),
        "up_proj": ("gate_up_proj", 1),
    }

    def __init__(self, config):
        super().__init__()
        ops_seq.load_if_built()                 # (prompt steps' gate|up: here, not inside the first of them)
        _, size = tp.world()
        self.geo = model_geometry(config, size)
        self.model = Qwen3Model(config, self.geo)
        self.lm_head = ParallelLMHead(config.vocab_size, config.hidden_size)
        if self.geo["tie"]:
            self.lm_head.weight.data = self.model.embed_tokens.weight.data

    @plain_calls
    def forward(self, input_ids: torch.Tensor, positions: torch.Tensor) -> torch.Tensor:
        return self.model(input_ids, positions)

    @plain_calls
    def compute_logits(self, hidden_states: torch.Tensor) -> torch.Tensor:
        return self.lm_head(hidden_states)

    def compute_logits_shard(self, hidden_states: torch.Tensor) -> torch.Tensor:
        """This rank's vocabulary slice of the logits (TP > 1: sampled shard-wise, never gathered)."""
        return self.lm_head.forward_shard(hidden_states)
