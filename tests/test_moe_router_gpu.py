"""The router kernel (logits, scores, choices and weights in one launch) against float64 logits and the route kernel on them: every number of entry
blocks and row blocks, ragged ends, group limits, correction, bias, the shared gate, both score forms and types, and rows that are not finite."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(1, 64, 1, 0, 1, 1, 1), (17, 192, 16, 1, 2, 1, 1), (64, 1024, 32, 1, 3, 4, 2), (65, 576, 33, 0, 4, 1, 1), (200, 128, 48, 0, 8, 6, 3),
         (33, 4096, 63, 1, 6, 9, 2), (3, 2112, 20, 1, 2, 1, 1), (600, 1536, 8, 0, 2, 1, 1), (300, 256, 64, 0, 6, 1, 1), (4097, 128, 12, 0, 2, 4, 2), (4130, 320, 30, 1, 3, 1, 1), (5000, 192, 40, 1, 3, 4, 2),
         (4099, 64, 60, 1, 4, 60, 7)]                 # rows, k, entries, gate, choices, groups, groups kept


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sigmoid,renorm,biased", [(False, True, False), (True, False, True), (True, True, False)])
@pytest.mark.parametrize("n,k,total,gate,top,count,keep", CASES)
def test_choices_and_weights(dtype, sigmoid, renorm, biased, n, k, total, gate, top, count, keep):
    from nano_vllm_amd import ops_seq
    g = torch.Generator(device="cuda").manual_seed(n + 7 * k + total)
    x = torch.randn(n, k + 8, generator=g, device="cuda").to(dtype)[:, :k]
    router = torch.randn(total + gate, k, generator=g, device="cuda") / k ** 0.5 * torch.logspace(-2, 0.5, total + gate, device="cuda").unsqueeze(1)
    bias = torch.randn(total + gate, generator=g, device="cuda") if biased else None
    correction = 0.05 * torch.randn(total, generator=g, device="cuda")
    ids, wts, got_gate = ops_seq.moe_router(x, router, bias, total, correction, top, count, keep, 1.5, sigmoid, renorm)
    z = x.double() @ router.double().T + (bias.double() if biased else 0)
    # sums of k exact or once rounded products in 32 bits: 4 sqrt(k) roundings of the largest logit's size
    tol = 4 * k ** 0.5 * 2.0 ** -24 * float(z.abs().max()) + 1e-7
    if gate:
        assert got_gate.shape == (n, 1) and float((got_gate[:, 0].double() - z[:, total]).abs().max()) <= tol
    else:
        assert got_gate is None
    s = torch.sigmoid(z[:, :total]) if sigmoid else torch.softmax(z[:, :total], 1)
    c = s + correction.double()
    close = torch.zeros(n, dtype=torch.bool, device="cuda")         # rows whose choices hang on less than the logits' error
    if count > 1:
        per = c.view(n, count, total // count).max(2).values
        order = per.sort(1, descending=True)
        if keep < count:
            close |= order.values[:, keep - 1] - order.values[:, keep] < 4 * tol
        out = torch.ones(n, count, dtype=torch.bool, device="cuda").scatter_(1, order.indices[:, :keep], False)
        c = c.masked_fill(out.repeat_interleave(total // count, 1), float("-inf"))
    best = c.sort(1, descending=True)
    for i in range(min(top, total - 1)):
        close |= (best.values[:, i] - best.values[:, i + 1] < 4 * tol) & torch.isfinite(best.values[:, i + 1])
    want = best.indices[:, :top]
    ok = ~close
    assert n < 8 or float(ok.float().mean()) > 0.6
    assert bool((ids.long()[ok] == want[ok]).all())
    w = s.gather(1, want)
    w = w / w.sum(1, keepdim=True) * 1.5 if renorm else w * 1.5
    assert float(((wts.double() - w)[ok].abs() / w[ok].clamp(min=1e-3)).max()) <= 4 * tol + 4e-6


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_that_are_not_finite_stay_alone(dtype):
    from nano_vllm_amd import ops_seq
    g = torch.Generator(device="cuda").manual_seed(3)
    x, router = torch.randn(40, 256, generator=g, device="cuda").to(dtype), torch.randn(20, 256, generator=g, device="cuda")
    ids, wts, _ = ops_seq.moe_router(x, router, None, 20, None, 4, 1, 1, 1.0, True, False)
    y = x.clone()
    y[7, 100], y[30, 3] = float("inf"), float("nan")
    ids2, wts2, _ = ops_seq.moe_router(y, router, None, 20, None, 4, 1, 1, 1.0, True, False)
    same = torch.ones(40, dtype=torch.bool, device="cuda")
    same[7] = same[30] = False
    assert bool((ids[same] == ids2[same]).all()) and bool((wts[same] == wts2[same]).all())
    assert bool(((ids2 >= 0) & (ids2 < 20)).all())
    # an infinity makes every logit one of both signs: entries with a positive weight there score 1, the first four of them are chosen
    first = (router[:, 100] > 0).nonzero()[:4, 0]
    assert bool((ids2[7].long() == first).all()) and bool((wts2[7] == 1.0).all())
