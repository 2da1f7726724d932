"""The 32-bit attention kernel on the matrix cores (csrc/seq/attn_f32.hip) against the scalar kernel, which takes every call: portions around its tiles of 16
columns and 16 keys, 1 to 20 heads over a kv head, all masks, sinks, norms, rotations, gates, caps and pooled blocks, and values that are not finite."""
import pytest
import torch

pytestmark = pytest.mark.gpu

PAGE = 64


def call(scalar, H, G, d, dv, lens, ctx, window=0, chunk=0, rot=0, norm="", sink=False, gate=0, temp=None, pool=0, cap=0.0, seed=0, page=PAGE, spoil=None):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g)
    n, total = sum(lens), [a + b for a, b in zip(lens, ctx)]
    need = [-(-t // page) for t in total]
    ids = torch.randperm(sum(need) + 2, generator=g)[:sum(need)].split(need)
    table = torch.full((len(lens), max(need) + 1), -1, dtype=torch.int32)
    pages = sum(need) + 2
    k, v = rand(pages, page, G, d), rand(pages, G, dv, page)
    for row, (mine, t) in enumerate(zip(ids, total)):
        table[row, :len(mine)] = mine.to(torch.int32)
        if t % page:                                        # what an earlier request left behind the end
            k[mine[-1], t % page:] = float("nan")
            v[mine[-1], :, :, t % page:] = float("inf")
        for j in spoil or ():                               # a token's own values
            if j < t:
                v[mine[j // page], :, 3, j % page] = float("inf")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    por = ops_seq.Portions(i32([0] + lens).cumsum(0).to(torch.int32), i32(ctx), i32(list(range(len(lens)))),
                           torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens)).to(torch.int32).cuda(), len(lens), n, max(lens))
    q = rand(n, H * d + 4).cuda()[:, :H * d]
    w = (1 + 0.1 * rand(H * d if norm == "rows" else d)).cuda() if norm else None
    kw = dict(gate_per_head=gate == 1, sink=rand(H).cuda() if sink else None, q_temp=temp, softcap=cap)
    if norm == "rows":
        kw["q_row"] = (0.5 + torch.rand(n, generator=g)).cuda()
    if pool:
        rows = ops_seq.pool_rows(page, pool)
        kw.update(pool=pool, pool_k=rand(pages, rows, G, d).cuda(), pool_v=rand(pages, rows // 8, G, dv, 8).cuda())
    gates = rand(n, H * (1 if gate == 1 else dv)).cuda() if gate else None
    freq = (1000.0 ** (-torch.arange(rot // 2) / max(rot // 2, 1))).float().cuda() if rot else None
    out = torch.full((n, H * dv), 9.0, device="cuda")
    lib = ops_seq.load_library()
    lib.nvs_window_attn_force_scalar(1 if scalar else 0)
    try:
        ops_seq.window_attn(q, w, 1e-6, gates, k.cuda().view(pages * page, G, d), v.cuda().view(pages * page, G, dv), table.cuda(), page, por, H, G, d, dv,
                            d ** -0.5, window, out, chunk, freq, **kw)
    finally:
        lib.nvs_window_attn_force_scalar(0)
    return out


CASES = [
    dict(H=4, G=2, lens=[1, 7, 8, 9, 15, 16, 17, 33, 65], ctx=[0] * 9),
    dict(H=2, G=2, lens=[20, 40, 9], ctx=[63, 64, 1], window=33, sink=True, page=16),
    dict(H=3, G=1, lens=[50, 70], ctx=[0, 130], chunk=48, rot=128, norm="head"),
    dict(H=8, G=1, lens=[100], ctx=[5], window=64, gate=2, temp=(0.3, 16)),
    dict(H=40, G=2, lens=[15, 14], ctx=[100, 0], rot=40, gate=1, sink=True),
    dict(H=4, G=2, lens=[90, 6], ctx=[0, 333], window=40, pool=4, cap=5.0, norm="rows", sink=True),
    dict(H=4, G=4, lens=[50, 14], ctx=[700, 0], window=64, pool=16, cap=30.0, norm="rows", rot=64),
    dict(H=1, G=1, lens=[1] * 70, ctx=[7 * i for i in range(70)]),
    dict(H=16, G=1, lens=[1] * 5, ctx=[0, 15, 16, 400, 1300], window=1024, page=256),
]


@pytest.mark.parametrize("d,dv", [(128, 128), (256, 192)])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_agrees_with_the_scalar_kernel(d, dv, case):
    kw = dict(CASES[case], d=d, dv=dv, seed=case)
    got, want = call(False, **kw).double(), call(True, **kw).double()
    assert torch.isfinite(want).all()
    # both keep 32 bits throughout: sums of d and of some hundred keys in another order
    assert ((got - want).norm() / want.norm()).item() <= 1e-6
    assert ((got - want).abs().max() / want.pow(2).mean().sqrt()).item() <= 3e-5


@pytest.mark.parametrize("d,dv", [(128, 128), (256, 192)])
@pytest.mark.parametrize("window,chunk", [(20, 0), (0, 24), (0, 0)])
def test_values_that_are_not_finite_reach_who_sees_them(d, dv, window, chunk):
    kw = dict(H=4, G=2, lens=[70, 33], ctx=[0, 20], window=window, chunk=chunk, d=d, dv=dv, spoil=(5, 30, 41))
    got, want = call(False, **kw), call(True, **kw)
    assert torch.equal(torch.isfinite(got), torch.isfinite(want)) and not torch.isfinite(want).all() and torch.isfinite(want).any()
    ok = torch.isfinite(want)
    assert ((got - want)[ok].double().norm() / want[ok].double().norm()).item() <= 1e-6
