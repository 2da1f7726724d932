"""Products in tiles of 256 rows (csrc/seq/gemm_tiles.h) where they can go wrong: one row and one feature unit, the edges of a tile in rows and features, the fewest
steps (two) and counts that leave the ring at each of its places, passes that are whole, part-filled above half (whole tiles) and below (halves of 128 rows), and
plans with experts of no row, half a tile and one row more."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def products(x, w):
    """x w^T in 64 bits, and what a sum of K products in 32 bits, in any order, may be off by: K 2^-24 of the sum of their sizes."""
    x, w = x.double(), w.double()
    return x @ w.T, x.shape[1] * 2.0 ** -24 * (x.abs() @ w.abs().T)


def every_value(got, want, off):
    """No value is off by more than `off` and one rounding to bfloat16 (half a step of 8 bits: 2^-8 of a value at most): a lost or stale 16-byte unit among millions
    does not show in a norm."""
    wrong = ((got.double() - want).abs() > 2.0 ** -8 * want.abs() + off * (1 + 2.0 ** -8)).sum().item()
    assert wrong == 0, f"{wrong} of {want.numel()} values"


def gated(y, off, ff):
    """silu(g) u and its bound: SiLU's slope is below 1.1, its own error and the product's below 2^-21."""
    g, u, eg, eu = y[:, :ff], y[:, ff:], off[:, :ff], off[:, ff:]
    a = torch.nn.functional.silu(g)
    return a * u, 1.1 * eg * (u.abs() + eu) + a.abs() * eu + 2.0 ** -21 * (a * u).abs()


@pytest.mark.parametrize("n,ff,K", [(1, 8, 128), (128, 128, 192), (129, 136, 256), (257, 1000, 320), (256, 256, 384), (2048, 4096, 128), (2100, 4096, 192),
                                    (3072, 4096, 448), (3100, 4096, 128), (9000, 768, 1024)])
def test_dense_products(n, ff, K):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(n + ff)
    x = torch.randn(n, K + 8, generator=g).to(torch.bfloat16).cuda()[:, :K]
    w = (torch.randn(2 * ff, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
    room = torch.full((n + 300, ff + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    want, off = gated(*products(x, w), ff)
    before = None
    for _ in range(2):
        ops_seq.silu_linear(x, w, 256, room[:n, :ff])
        # one rounding of the result to bfloat16, 2^-9 at most per value
        assert ((room[:n, :ff].double() - want).norm() / want.norm()).item() <= 2.0 ** -8
        assert (room[n:] == 7.0).all() and (room[:, ff:] == 7.0).all()
        every_value(room[:n, :ff], want, off)
        assert before is None or torch.equal(before, room)          # (the order of a sum is fixed)
        before = room.clone()


@pytest.mark.parametrize("biased", [False, True])
@pytest.mark.parametrize("n,N,K", [(1, 8, 128), (128, 264, 192), (257, 1000, 320), (4096, 4096, 128), (4100, 4096, 192), (6144, 4096, 128), (6200, 4104, 256)])
def test_dense_rows(n, N, K, biased):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(n + N)
    x = torch.randn(n, K + 8, generator=g).to(torch.bfloat16).cuda()[:, :K]
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
    b = torch.randn(N, generator=g).to(torch.bfloat16).cuda() if biased else None
    room = torch.full((n + 300, N + 8), 7.0, dtype=torch.bfloat16, device="cuda")
    want, off = products(x, w)
    if biased:
        want, off = want + b.double(), off + 2.0 ** -24 * (want.abs() + b.double().abs())
    before = None
    for _ in range(2):
        ops_seq.linear_tiles(x, w, b, room[:n, :N])
        assert ((room[:n, :N].double() - want).norm() / want.norm()).item() <= 2.0 ** -8          # (one rounding of the result to bfloat16)
        assert (room[n:] == 7.0).all() and (room[:, N:] == 7.0).all()
        every_value(room[:n, :N], want, off)
        assert before is None or torch.equal(before, room)
        before = room.clone()


@torch.inference_mode()
@pytest.mark.parametrize("n,N,K", [(2900, 2576, 192), (13550, 1024, 256), (800, 12288, 512)])
def test_linear_layers_take_the_tiles_where_the_rule_says(n, N, K):
    from nano_vllm_amd import ops_seq
    from nano_vllm_amd.layers import ReplicatedLinear
    layer = ReplicatedLinear(K, N, bias=True).to(torch.bfloat16).cuda()
    layer.weight.data.copy_(torch.randn(N, K) / K ** 0.5)
    layer.bias.data.copy_(torch.randn(N))
    x = torch.randn(n, K).to(torch.bfloat16).cuda()
    assert ops_seq.many_rows(x, layer.weight, layer.bias)
    want = x.double() @ layer.weight.double().T + layer.bias.double()
    for got in (layer(x), ops_seq.linear(x, layer.weight.data, layer.bias.data)):
        assert ((got.double() - want).norm() / want.norm()).item() <= 2.0 ** -8
    with torch.inference_mode(False):
        assert not ops_seq.many_rows(x, layer.weight, layer.bias)               # (somebody may differentiate)


@pytest.mark.parametrize("mode", ["glu", "relu2", "rows"])
@pytest.mark.parametrize("counts,nout,K", [([0, 1, 256, 257, 128, 129], 264, 128), ([5], 8, 192), ([700, 0, 0, 513], 8192, 256), ([2300, 1, 1000], 4096, 320)])
def test_grouped_products(mode, counts, nout, K):
    from nano_vllm_amd import ops_seq
    E, n = len(counts), sum(counts)
    g = torch.Generator().manual_seed(nout + K)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(n, generator=g)].to(torch.int32).cuda()
    x = torch.randn(n, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(E, (2 if mode == "glu" else 1) * nout, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
    plan = ops_seq.moe_plan(ids.view(n, 1), E, 256)
    rows = plan.pair_row.view(-1).long()
    src = x
    if mode == "rows":
        src = torch.full((plan.cap, K), float("nan"), dtype=torch.bfloat16, device="cuda")
        src[rows] = x
    out = torch.full((plan.cap, nout), 7.0, dtype=torch.bfloat16, device="cuda")
    before = None
    for _ in range(2):
        ops_seq.moe_gemm(src, w, plan, mode == "glu", out, relu2=mode == "relu2")
        assert before is None or torch.equal(before, out)
        before = out.clone()
    for e in range(E):
        mine = (ids == e).nonzero().view(-1)
        if not len(mine):
            continue
        y, off = products(x[mine], w[e])
        if mode == "glu":
            want, off = gated(y, off, nout)
        elif mode == "relu2":                                       # (the square is one more rounding)
            want, off = y.clamp(min=0) ** 2, 2 * y.abs() * off + off ** 2 + 2.0 ** -23 * y ** 2
        else:
            want = y
        assert ((out[rows[mine]].double() - want).norm() / want.norm()).item() <= 2.0 ** -8       # (one rounding of the result to bfloat16)
        every_value(out[rows[mine]], want, off)
    untouched = torch.ones(plan.cap, dtype=torch.bool, device="cuda")
    untouched[rows] = False
    assert (out[untouched] == 7.0).all()
