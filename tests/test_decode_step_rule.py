"""When a decode step's layers go in one launch (Qwen3Model._decode_step), seen on the CPU: layers as the file makes them do, and layers of which anything is watched, replaced or
extended, in an instance or in its class, are called as they are; nothing is read of a module that is somebody else's."""
from types import SimpleNamespace

import pytest
import torch
from torch import nn

from nano_vllm_amd import layers, ops, qwen3


@pytest.fixture
def model(monkeypatch):
    monkeypatch.setattr(layers, "_rope_singleton", lambda h, r, n, base, device: rope)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    rope = layers.RotaryEmbedding(128, 128, 64, 1e6)
    config = SimpleNamespace(hidden_size=1024, intermediate_size=1024, num_hidden_layers=2, num_attention_heads=8, num_key_value_heads=4, head_dim=128, rms_norm_eps=1e-6,
                             vocab_size=16, hidden_act="silu", max_position_embeddings=64, rope_theta=1e6, tie_word_embeddings=True, attention_bias=False)
    torch.set_default_dtype(torch.bfloat16)
    try:
        m = qwen3.Qwen3ForCausalLM(config).model
    finally:
        torch.set_default_dtype(torch.float32)
    for layer in m.layers:
        layer.self_attn.attn.k_cache, layer.self_attn.attn.v_cache = (torch.zeros(2, 4, 32, 128, dtype=torch.bfloat16) for _ in range(2))
    calls = []
    monkeypatch.setattr(ops, "decode_step_bytes", lambda rows, *a: 256)
    monkeypatch.setattr(ops, "paged_attn_decode_workspace_bytes", lambda *a: 256)
    monkeypatch.setattr(ops, "decode_step", lambda x, tensors, *a, **k: calls.append(tensors) or "both")
    monkeypatch.setattr(qwen3, "get_context", lambda: SimpleNamespace(
        is_prefill=False, shared_prefix=False, context_lens=torch.ones(2, dtype=torch.int32), block_tables=torch.zeros(2, 2, dtype=torch.int32), decode_workspace=None,
        max_context=64, decode_gave_up=None))

    class Rows:                                    # a step's rows, on a GPU as far as anybody asks
        shape, dtype, is_cuda = (2, 1024), torch.bfloat16, True
        dim = staticmethod(lambda: 2)
        is_contiguous = staticmethod(lambda: True)
    return m, calls, Rows()


def test_layers_as_made_go_in_one_launch(model):
    m, calls, x = model
    assert m._decode_step(x) == "both"
    for layer, tensors in zip(m.layers, calls[0]):
        a, f = layer.self_attn, layer.mlp
        want = (layer.input_layernorm.weight, a.qkv_proj.weight, a.q_norm.weight, a.k_norm.weight, a.o_proj.weight, layer.post_attention_layernorm.weight,
                f.gate_up_proj.weight, f.down_proj.weight, a.attn.k_cache, a.attn.v_cache)
        assert len(tensors) == 10 and all(s is t for s, t in zip(tensors, want))


class Wrapped(nn.Module):
    """Somebody's own projection: what a decode step calls of it, and nothing else."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward_decode(self, x):
        return self.inner.forward_decode(x)


class Bare(nn.Module):
    def forward(self, x, residual=None):
        return x, residual


class Pruned(qwen3.Qwen3MLP):
    pass


def narrower(layer):
    layer.mlp.gate_up_proj.weight, layer.mlp.down_proj.weight = (nn.Parameter(torch.zeros(s, dtype=torch.bfloat16), requires_grad=False) for s in ((1024, 1024), (1024, 512)))


def plain_bias(layer):
    del layer.self_attn.o_proj._parameters["bias"]
    layer.self_attn.o_proj.bias = torch.ones(1024, dtype=torch.bfloat16)


def askew(layer):
    layer.mlp.down_proj.weight = nn.Parameter(torch.zeros(1024 * 1024 + 4, dtype=torch.bfloat16)[4:].view(1024, 1024), requires_grad=False)


CHANGES = dict(
    wrapped=lambda l: setattr(l.mlp, "down_proj", Wrapped(l.mlp.down_proj)), norm=lambda l: setattr(l, "input_layernorm", Bare()), norm2=lambda l: setattr(l, "post_attention_layernorm", Bare()),
    attention=lambda l: setattr(l.self_attn, "attn", Bare()), whole=lambda l: setattr(l, "self_attn", Bare()), mlp=lambda l: setattr(l, "mlp", Bare()),
    subclass=lambda l: setattr(l.mlp, "__class__", Pruned), own_call=lambda l: setattr(l.mlp.down_proj, "forward_decode", lambda x: x), hook=lambda l: l.self_attn.o_proj.register_forward_hook(print),
    narrower=narrower, plain_bias=plain_bias, askew=askew, wide=lambda l: setattr(l.mlp.down_proj, "weight", nn.Parameter(l.mlp.down_proj.weight.float(), requires_grad=False)),
    no_activation=lambda l: None)


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("change", list(CHANGES))
def test_layers_that_are_somebody_s_own_are_called(model, change, which):
    m, calls, x = model
    CHANGES[change](m.layers[which])
    if change == "no_activation":                  # (nothing of a decode step calls it)
        del m.layers[which].mlp.act_fn
        assert m._decode_step(x) == "both"
        return
    assert m._decode_step(x) is None and not calls


@pytest.mark.parametrize("kind,name", [(qwen3.Qwen3MLP, "forward"), (qwen3.Qwen3MLP, "forward_normed"), (qwen3.Qwen3Attention, "forward"), (qwen3.Qwen3DecoderLayer, "forward"),
                                       (layers.RMSNorm, "forward"), (layers.RMSNorm, "into_linear"), (layers.Attention, "forward_open"), (layers.LinearBase, "forward"),
                                       (layers.RowParallelLinear, "forward_decode"), (layers.MergedColumnParallelLinear, "forward_silu"), (nn.Module, "__call__")])
def test_a_call_that_is_replaced_in_its_class_is_made(model, monkeypatch, kind, name):
    m, calls, x = model
    kept = getattr(kind, name)
    monkeypatch.setattr(kind, name, lambda *a, **k: kept(*a, **k))
    assert m._decode_step(x) is None and not calls
