"""A routed layer's rows summed by the norm behind it: the bits of the sum and the norm as launches of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _parts(n, width, top, dtype, shared, gate, passing, g):
    """Rows in a plan's order with gaps, as expert tiles leave them; some choices without a row."""
    from types import SimpleNamespace
    rows = torch.randn(2 * n * top + 3, width + 8, generator=g).to(dtype).cuda()[:, :width]
    pair = torch.randperm(rows.shape[0], generator=g)[:n * top].view(n, top).int()
    if passing:
        pair[torch.rand(n, top, generator=g) < 0.3] = -1
    wts = torch.rand(n, top, generator=g).cuda()
    h = torch.randn(n, width + 4, generator=g).to(dtype).cuda()[:, :width]
    sh = torch.randn(n, width, generator=g).to(dtype).cuda() if shared else None
    z = torch.randn(n, 5, generator=g).cuda()[:, 4:] if gate else None
    return h, rows, SimpleNamespace(pair_row=pair.cuda()), wts, sh, z


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,width,top,shared,gate,passing", [
    (3, 4, 1, False, False, False), (70, 64, 3, True, True, True), (5, 1000, 5, True, False, False), (33, 1024, 4, False, False, False), (9, 1028, 6, True, True, True),
    (600, 2048, 4, True, True, False), (515, 4096, 3, True, False, True), (513, 8192, 2, True, True, True)])
def test_sums_and_norms_in_one_pass(dtype, n, width, top, shared, gate, passing):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(n + width)
    parts = _parts(n, width, top, dtype, shared, gate, passing, g)
    chosen = ops_seq.ChosenRows(*parts)
    w, wa = (torch.randn(width, generator=g).to(dtype).cuda() for _ in range(2))
    x0 = torch.randn(n, width, generator=g).cuda()
    assert chosen.fits(x0, w, wa)
    h, rows, plan, wts, sh, z = parts
    y = torch.empty(n, width, dtype=dtype, device="cuda")
    ops_seq.moe_combine(rows, plan, wts, h, sh, z, y)
    for center in (False, True):
        for weight in (w, None):
            got, want = [], []
            for a, res in ((chosen, got), (y, want)):
                x, out = x0.clone(), torch.empty_like(y) if weight is not None else None
                ops_seq.add_group_norm(x, weight, 1, 1e-6, out, a=a, a_mult=0.75, center=center)
                res += [x, out]
            assert torch.equal(got[0], want[0]) and (weight is None or torch.equal(got[1], want[1])), (center, weight is None)
    for weight in (w, None):
        got, want = [], []
        for a, res in ((chosen, got), (y, want)):
            x, out = x0.clone(), torch.empty_like(y) if weight is not None else None
            ops_seq.sandwich_norm(x, a, wa, weight, 1e-6, out, a_mult=0.75)
            res += [x, out]
        assert torch.equal(got[0], want[0]) and (weight is None or torch.equal(got[1], want[1])), weight is None
    # choices beside another output, whose norm is scaled (choices without a row are left out there)
    x, y64 = x0.clone(), torch.zeros(n, width, dtype=torch.float64)
    for t in range(n):
        for k in range(top):
            r = int(plan.pair_row[t, k])
            if r >= 0:
                y64[t] += wts[t, k].double().cpu() * rows[r].double().cpu()
    if sh is not None:
        y64 += sh.double().cpu()
    ops_seq.branch_norm(x, sh, w, None, 1e-6, None, (rows, plan, wts))
    want = x0.double().cpu() + y64 / (y64.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * w.double().cpu()
    assert ((x.double().cpu() - want).abs().max() <= 1e-5 * want.abs().max()).item()          # (sums in 32 bits of what 16 or 32 bits hold)


def test_what_the_pass_does_not_take_is_summed_first():
    """Groups, a second addend, widths that are no whole accesses, few wide rows: the launches of their own, with their results."""
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(1)
    for width, groups, second in ((64, 4, False), (64, 1, True), (66, 1, False), (65, 1, False), (2052, 1, False)):
        parts = _parts(7, width, 2, torch.bfloat16, True, True, True, g)
        chosen = ops_seq.ChosenRows(*parts)
        w = torch.randn(width, generator=g).bfloat16().cuda()
        x0, b = torch.randn(7, width, generator=g).cuda(), torch.randn(7, width, generator=g).cuda() if second else None
        h, rows, plan, wts, sh, z = parts
        y = torch.empty(7, width, dtype=torch.bfloat16, device="cuda")
        ops_seq.moe_combine(rows, plan, wts, h, sh, z, y)
        got, want = [], []
        for a, res in ((chosen, got), (y, want)):
            x, out = x0.clone(), torch.empty_like(y)
            ops_seq.add_group_norm(x, w, groups, 1e-6, out, a=a, b=b)
            res += [x, out]
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), (width, groups, second)
