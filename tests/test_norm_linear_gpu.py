"""A linear layer of few rows with the residual add and norm in front (nvl_norm_linear) against float64 on the same bfloat16 inputs, at the edges of its row
and column blocks and for reductions that give some wavefronts no piece."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def rand(g, *s, scale=1.0):
    return (scale * torch.randn(*s, generator=g, device="cuda")).bfloat16()


def rel(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 4, 64), (1, 4096, 1024), (2, 36, 192), (8, 3072, 1024), (9, 1000, 576), (15, 68, 2048), (16, 1024, 2048), (3, 24, 1088)])
@pytest.mark.parametrize("first,slabs", [(False, 0), (True, 0), (False, 1), (False, 2), (False, 4), (True, 4)])
def test_norm_and_layer(m, n, k, silu, first, slabs):
    from nano_vllm_amd import ops
    g = torch.Generator(device="cuda").manual_seed(m * 1000 + n + k)
    x, r, nw = rand(g, m, k) if not slabs else torch.randn(slabs, m, k, generator=g, device="cuda"), None if first else rand(g, m, k, scale=3.0), (1 + 0.1 * torch.randn(k, generator=g, device="cuda")).bfloat16()
    w = rand(g, n * (2 if silu else 1), k, scale=k ** -0.5)
    before = None if first else r.clone()
    out, new = ops.norm_linear(x, r, nw, 1e-6, w, silu)
    if slabs:                                                       # summed in order, rounded once
        x = sum(x[i] for i in range(1, slabs)) + x[0] if slabs < 3 else ((x[0] + x[1]) + x[2]) + x[3]
        x = x.bfloat16()
    s = x.double() + (0 if first else before.double())
    assert first or torch.equal(r, before)
    assert torch.equal(new, (x.float() + (0 if first else before.float())).bfloat16())
    h = (s * torch.rsqrt((s * s).mean(1, keepdim=True) + 1e-6) * nw.double())
    z = h.float().bfloat16().double() @ w.double().T
    want = torch.nn.functional.silu(z[:, :n]) * z[:, n:] if silu else z
    # the layer's input and its result are rounded to 8 bits (a norm in 32 bits may round an entry to the neighbour); with SiLU gate and up too
    assert rel(out, want) <= 2.0 ** -8 * (2 if silu else 1)


def test_what_is_not_covered_is_refused():
    from nano_vllm_amd import ops
    x, w = torch.zeros(17, 64, device="cuda").bfloat16(), torch.zeros(64, 64, device="cuda").bfloat16()
    with pytest.raises(ops.NvlError, match="up to 16 rows"):
        ops.norm_linear(x, None, w[0], 1e-6, w)


@pytest.mark.parametrize("rows,width,taken", [(1, 1024, True), (8, 1024, True), (9, 1024, False), (16, 1024, False), (1, 2048, False), (8, 512, True)])
def test_layer_takes_it_where_it_pays(rows, width, taken):
    from nano_vllm_amd.layers import QKVParallelLinear, RMSNorm
    norm = RMSNorm(width).to(torch.bfloat16).cuda()
    qkv = QKVParallelLinear(width, 128, 16, 8, bias=False).to(torch.bfloat16).cuda()
    both = norm.into_linear(torch.ones(rows, width, device="cuda").bfloat16(), None, qkv)
    assert (both is not None) == taken
