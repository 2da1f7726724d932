"""The real-gated linear recurrence: gates over their whole range against a token loop in float64, portions around the eight tokens whose
operands are asked for together and portions cut into segments; a NaN in any operand stays visible, in its channel and from its token on."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def _portions(lens, ctx):
    from nano_vllm_amd.ops_seq import Portions
    i = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return Portions(i(cu), i(ctx), i(range(len(lens))), i([s for s, n in enumerate(lens) for _ in range(n)]), len(lens), cu[-1], max(lens))


def _inputs(lens, channels, seed, spread=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, blocks = sum(lens), 4
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    # (a gate of e^-87 and less is no normal 32-bit number any more)
    return dict(gates=(spread * rand(blocks, n, 2 * channels // blocks)).clamp(-80, 80), u=rand(n, channels), ypre=rand(n, channels), lam=rand(channels)), rand(len(lens), channels)


def _run(x, S, lens, ctx):
    from nano_vllm_amd import ops_seq
    S, out = S.clone(), torch.empty_like(x["u"])
    ops_seq.rglru_scan(x["gates"], x["u"], x["ypre"], x["lam"], 8.0, x["gates"].shape[0], _portions(lens, ctx), S, out)
    return out, S


@pytest.mark.parametrize("spread", [1.0, 30.0])
@pytest.mark.parametrize("lens", [[1, 7, 3], [1, 7, 8, 9, 17], [700, 3, 64]], ids=["few", "short", "segments"])
def test_against_the_token_loop(lens, spread):
    channels, ctx = 64, [5 * (s % 2) for s in range(len(lens))]
    x, S = _inputs(lens, channels, 3, spread)
    got, end = _run(x, S, lens, ctx)
    n, F = sum(lens), torch.float64
    gates = x["gates"].to(F).view(4, n, 2, channels // 4).permute(2, 1, 0, 3).reshape(2, n, channels)
    la = -8.0 * torch.sigmoid(gates[0]) * torch.nn.functional.softplus(x["lam"].to(F))
    a, add = la.exp(), (-torch.expm1(2 * la)).sqrt() * torch.sigmoid(gates[1]) * x["u"].to(F)
    gelu = torch.nn.functional.gelu(x["ypre"].to(F), approximate="tanh")
    at = 0
    for s, ln in enumerate(lens):
        st = S[s].to(F) * (ctx[s] > 0)
        err = torch.zeros_like(st)
        for t in range(at, at + ln):
            # log a is a sigmoid, a softplus and two products of 2^-24 to 2^-23 each: a is off by eight times that much of |log a|, and by its own
            # rounding; the added term by a dozen roundings; the update by one. A segment's decay is the exponential of a sum of logarithms.
            err = a[t] * err + EPS * ((8 * la[t].abs() + 3) * a[t] * st.abs() + 12 * add[t].abs())
            st = a[t] * st + add[t]
            tol = (err + 8 * EPS * st.abs()) * gelu[t].abs() + 8 * EPS * st.abs() * x["ypre"][t].abs()
            assert ((got[t].to(F) - st * gelu[t]).abs() <= tol + 1e-37).all(), (s, t - at)
        assert ((end[s].to(F) - st).abs() <= err + 8 * EPS * st.abs() + 1e-37).all(), s
        at += ln


@pytest.mark.parametrize("operand", ["recurrence gate", "input gate", "u", "ypre", "lam", "state"])
@pytest.mark.parametrize("lens,seq,j", [([1, 7, 2], 1, 3), ([3, 21, 9], 1, 12), ([900, 5], 0, 333)], ids=["few", "whole", "segments"])
def test_a_nan_stays_visible(lens, seq, j, operand):
    channels, c, ctx = 32, 13, [2] * len(lens)
    x, S = _inputs(lens, channels, 5)
    clean, end = _run(x, S, lens, ctx)
    first = sum(lens[:seq])
    token = first + j
    nan, bad, bad_end = float("nan"), torch.zeros_like(clean, dtype=torch.bool), torch.zeros_like(end, dtype=torch.bool)
    bw = channels // 4
    if operand.endswith("gate"):
        x["gates"][c // bw, token, c % bw + (bw if operand == "input gate" else 0)] = nan
    elif operand == "lam":
        x["lam"][c] = nan
    elif operand == "state":
        S[seq, c] = nan
    else:
        x[operand][token, c] = nan
    if operand == "ypre":
        bad[token, c] = True
    elif operand == "lam":
        bad[:, c], bad_end[:, c] = True, True
    else:
        bad[first if operand == "state" else token:first + lens[seq], c], bad_end[seq, c] = True, True
    got, got_end = _run(x, S, lens, ctx)
    assert torch.equal(got.isnan(), bad) and torch.equal(got_end.isnan(), bad_end)
    assert torch.equal(got[~bad], clean[~bad]) and torch.equal(got_end[~bad_end], end[~bad_end])
