"""The real-gated linear recurrence: a NaN in any operand stays visible, in its channel and from its token on."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _portions(lens, ctx):
    from nano_vllm_amd.ops_seq import Portions
    i = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return Portions(i(cu), i(ctx), i(range(len(lens))), i([s for s, n in enumerate(lens) for _ in range(n)]), len(lens), cu[-1], max(lens))


def _inputs(lens, channels, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, blocks = sum(lens), 4
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    return dict(gates=rand(blocks, n, 2 * channels // blocks), u=rand(n, channels), ypre=rand(n, channels), lam=rand(channels)), rand(len(lens), channels)


def _run(x, S, lens, ctx):
    from nano_vllm_amd import ops_seq
    S, out = S.clone(), torch.empty_like(x["u"])
    ops_seq.rglru_scan(x["gates"], x["u"], x["ypre"], x["lam"], 8.0, x["gates"].shape[0], _portions(lens, ctx), S, out)
    return out, S


@pytest.mark.parametrize("operand", ["recurrence gate", "input gate", "u", "ypre", "lam", "state"])
@pytest.mark.parametrize("lens,seq,j", [([3, 21, 9], 1, 12), ([900, 5], 0, 333)], ids=["whole", "segments"])
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
