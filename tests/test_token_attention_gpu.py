"""The attention kernel for steps of single tokens (csrc/seq/attn_token.hip) against the scalar kernel, which takes every call: contexts around its tiles of
32 keys and the tiles its wavefronts take in turn, 1 to 40 heads over a kv head, all masks, sinks, norms, rotations, gates, temperatures and
caps, and places of the pages that are not seen and hold infinities and NaN."""
import pytest
import torch

from test_prompt_attention_gpu import SIZES, call, step

pytestmark = pytest.mark.gpu

CONTEXTS = [0, 1, 30, 31, 32, 33, 63, 64, 255, 256, 257, 511, 512, 700, 1300]
CASES = [
    dict(H=8, G=8),
    dict(H=4, G=2, window=33, sink=True),
    dict(H=6, G=2, window=64, rot=128, norm="head"),
    dict(H=40, G=2, chunk=48, rot=40, gate=1),                  # 20 heads over a kv head: two workgroups
    dict(H=16, G=1, window=1024, gate=2, temp=(0.3, 16)),
    dict(H=34, G=1, cap=5.0, sink=True),
    dict(H=4, G=4, cap=30.0, norm="rows", window=256, rot=64),
    dict(H=3, G=3, chunk=512, rot=128, norm="head", gate=2, sink=True, temp=(0.1, 64)),
]


@pytest.mark.parametrize("d,dv", SIZES)
@pytest.mark.parametrize("case", range(len(CASES)))
def test_single_tokens_agree_with_the_scalar_kernel(d, dv, case):
    kw = dict(CASES[case], lens=[1] * len(CONTEXTS), ctx=CONTEXTS, d=d, dv=dv, seed=case)
    got, want = call(False, **kw).double(), call(True, **kw).double()
    assert torch.isfinite(want).all()
    # both round the finished query and the result to 8 bits; the matrix cores round the weights too (2^-9 each, averaged over the keys)
    assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -7
    assert ((got - want).abs().max() / want.pow(2).mean().sqrt()).item() <= 0.1


@pytest.mark.parametrize("d,dv", SIZES)
@pytest.mark.parametrize("page", [32, 64, 256])
def test_weights_against_float64_and_values_before_the_window(d, dv, page):
    """Softmax in float64 on the same bfloat16 inputs: weights and result are rounded to 8 bits. Values that are not seen are not finite."""
    g = torch.Generator(device="cuda").manual_seed(page)
    H, G, window = 4, 2, 100
    ctx = [0, 40, 99, 100, 131, 400, 1001]
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    T = [c + 1 for c in ctx]
    K, V, q = rand(sum(T), G, d), rand(sum(T), G, dv), rand(len(ctx), H * d)
    want, at = [], 0
    for i, t in enumerate(T):
        lo = max(0, t - window)
        k, v = (x[at + lo:at + t].double().repeat_interleave(H // G, 1) for x in (K, V))
        w = torch.softmax(torch.einsum("hd,thd->ht", q[i].double().view(H, d), k) * d ** -0.5, 1)
        want.append(torch.einsum("ht,thv->hv", w, v))
        V[at:at + lo] = float("inf")
        K[at:at + lo, :, ::2] = float("nan")
        at += t
    got = step(q, K, V, [1] * len(ctx), ctx, H, G, d, dv, scale=d ** -0.5, window=window, page=page).view(len(ctx), H, dv).double()
    want = torch.stack(want)
    assert torch.isfinite(got).all()
    assert ((got - want).norm() / want.norm()).item() <= 2.0 ** -8
