"""The matrix-state recurrences in chunks of 16 tokens on 32-bit matrix instructions (state sizes 64 and 128) against a token loop in
float64: portions at the edges of a chunk and of the four chunks whose weights are computed together, rows that do not fill a
wavefront or a workgroup, portions cut into segments, states kept from earlier calls, dirty slots."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def _portions(lens, ctx, slots):
    from nano_vllm_amd.ops_seq import Portions
    i = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    p = Portions.__new__(Portions)
    p.cu_q, p.ctx0, p.slot = i(cu), i(ctx), i(slots)
    p.tseq = i([s for s, n in enumerate(lens) for _ in range(n)])
    p.nseq, p.n, p.max_q = len(lens), cu[-1], max(lens)
    return p


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("lens", [[1, 3, 2], [1, 2] * 40, [1, 16, 17, 2], [63, 65, 15], [700, 20, 300]], ids=["few", "crowd", "short", "group", "segments"])
@pytest.mark.parametrize("form,heads,P,N,G", [(0, 16, 16, 64, 1), (2, 16, 24, 64, 1), (0, 4, 64, 128, 2), (0, 3, 40, 64, 1), (0, 2, 100, 128, 2), (1, 3, 128, 128, 1), (1, 2, 16, 64, 1),
                                              (2, 2, 128, 128, 1), (2, 3, 24, 64, 1), (2, 2, 72, 128, 1),
                                              (0, 2, 136, 64, 1), (0, 1, 256, 64, 1), (1, 2, 200, 64, 1)])        # (two workgroups of rows)
def test_chunked_recurrences_against_the_token_loop(form, heads, P, N, G, lens, dtype):
    from nano_vllm_amd import ops_seq
    g = torch.Generator(device="cuda").manual_seed(heads * P + N + form)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    n, nseq, F = sum(lens), len(lens), torch.float64
    rows = P + 1 if form == 2 else P
    ctx = [7 * (s % 2) for s in range(nseq)]                    # every other portion continues a sequence
    slots = [nseq - s for s in range(nseq)]                     # slot 0 is nobody's
    por = _portions(lens, ctx, slots)
    S, M = rand(nseq + 1, heads, rows, N), rand(nseq + 1, heads).abs()
    state = torch.stack([S[slots[s]].double() * (ctx[s] > 0) for s in range(nseq)])
    mx = torch.stack([M[slots[s]].double() * (ctx[s] > 0) for s in range(nseq)])
    S0, M0 = S[0].clone(), M[0].clone()
    y, den = torch.empty(n, heads * P, device="cuda"), torch.empty(n, heads, device="cuda")
    skip = torch.zeros(heads, device="cuda", dtype=dtype)
    if form == 0:
        xbc, proj = rand(n, heads * P + 2 * G * N), rand(n, heads + 5).to(dtype)
        bias, A_log, skip = (rand(heads) - 2).to(dtype), rand(heads).to(dtype), rand(heads).to(dtype)
        ops_seq.ssd_scan(xbc, proj, 3, bias, A_log, skip, heads, P, N, G, por, S, y)
        x, B, C = xbc.double().split([heads * P, G * N, G * N], 1)
        B, C = (t.reshape(n, G, N).repeat_interleave(heads // G, 1) for t in (B, C))
        step = torch.nn.functional.softplus(proj[:, 3:3 + heads].double() + bias.double())
        decay = torch.exp(-torch.exp(A_log.double()) * step)
    else:
        cols = [heads * P, heads * N, heads * N, 2 * heads]
        proj = rand(n, (sum(cols) + 7) // 8 * 8).to(dtype)
        x, B, C, gates = proj.double()[:, :sum(cols)].split(cols, 1)
        B, C = B.reshape(n, heads, N), C.reshape(n, heads, N)
    if form == 1:
        rate = torch.exp(-torch.linspace(0.003, 2.0, heads, device="cuda"))
        ops_seq.decay_scan(proj, 0, cols[0], cols[0] + cols[1], rate, heads, N, P, por, S, y)
        x, B, C = (torch.nn.functional.silu(t) for t in (x, B, C))
        step, decay = torch.ones(n, heads, dtype=F, device="cuda"), rate.double().expand(n, heads)
    if form == 2:
        ib, fb, at = rand(heads).to(dtype), (rand(heads) + 2).to(dtype), sum(cols[:3])
        ops_seq.gated_memory_scan(proj, 0, cols[0], cols[0] + cols[1], at, at + heads, ib, fb, 15.0, N ** -0.5, heads, N, P, por, S, M, y, den)
        C = C * N ** -0.5
        ig = 15 * torch.tanh((gates[:, :heads] + ib.double()) / 15)
        fg = torch.nn.functional.logsigmoid(15 * torch.tanh((gates[:, heads:] + fb.double()) / 15))
    x = x.reshape(n, heads, P)
    if form == 2:
        x = torch.cat([x, torch.ones(n, heads, 1, dtype=F, device="cuda")], 2)
    size = state.abs()                                          # the same recurrence on absolute values: what an error is measured by
    at = 0
    for s, ln in enumerate(lens):
        for t in range(at, at + ln):
            if form == 2:
                m = torch.maximum(fg[t] + mx[s], ig[t])
                a, w = torch.exp(fg[t] + mx[s] - m), torch.exp(ig[t] - m)
                mx[s] = m
            else:
                a, w = decay[t], step[t]
            new = (w[:, None] * x[t])[:, :, None] * B[t][:, None]
            state[s] = a[:, None, None] * state[s] + new
            size[s] = a[:, None, None] * size[s] + new.abs()
            out, mag = (state[s] * C[t][:, None]).sum(2), (size[s] * C[t][:, None].abs()).sum(2)
            # an entry is a sum over N products of state entries, each a sum over the tokens so far; one rounding per step, and a
            # handful per term for its gate, its decay and the products
            tol = (t - at + 1 + N + 32) * EPS
            if form == 2:
                q, lim = out[:, P], torch.exp(-mx[s])
                want = torch.maximum(q.abs(), lim) + 1e-6
                assert ((den[t] - want).abs() <= tol * (mag[:, P] + lim) + 4 * EPS * mx[s].abs() * lim).all(), (s, t - at)
                out, mag = out[:, :P], mag[:, :P]
            out, mag = out + skip.double()[:, None] * x[t][:, :P], mag + (skip.double()[:, None] * x[t][:, :P]).abs()
            assert ((y[t].view(heads, P) - out).abs() <= tol * mag).all(), (s, t - at)
        assert ((S[slots[s]] - state[s]).abs() <= (ln + 32) * EPS * size[s]).all(), s
        if form == 2:
            assert ((M[slots[s]] - mx[s]).abs() <= (ln + 4) * EPS * mx[s].abs().clamp(min=1)).all(), s
        at += ln
    assert torch.equal(S[0], S0) and torch.equal(M[0], M0)


def _scan(form, heads, P, N, por, S, M, x, y, den):
    """One call on prepared operands: x holds xbc / proj and the gates' parameters."""
    from nano_vllm_amd import ops_seq
    if form == 0:
        ops_seq.ssd_scan(x["xbc"], x["proj"], 0, x["bias"], x["A_log"], x["D"], heads, P, N, 1, por, S, y)
    elif form == 1:
        ops_seq.decay_scan(x["proj"], 0, heads * P, heads * (P + N), x["rate"], heads, N, P, por, S, y)
    else:
        at = heads * (P + 2 * N)
        ops_seq.gated_memory_scan(x["proj"], 0, heads * P, heads * (P + N), at, at + heads, x["ib"], x["fb"], 15.0, N ** -0.5, heads, N, P, por, S,
                                  M, y, den)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("form,heads,P,N", [(0, 2, 64, 128), (0, 2, 100, 64), (1, 2, 64, 64), (1, 2, 128, 128), (2, 2, 64, 64), (2, 2, 128, 128)])
@pytest.mark.parametrize("lens,seq,j", [([40, 70, 20], 1, 27), ([600, 9], 0, 301)], ids=["whole", "segments"])
def test_a_value_that_is_not_finite_reaches_no_earlier_token(lens, seq, j, form, heads, P, N, value):
    g = torch.Generator(device="cuda").manual_seed(P + form)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    n, nseq = sum(lens), len(lens)
    rows = P + (form == 2)
    x = dict(xbc=rand(n, heads * P + 2 * N), proj=rand(n, heads * (P + 2 * N) + 8), bias=rand(heads) - 2, A_log=rand(heads), D=rand(heads),
             rate=torch.full((heads,), 0.95, device="cuda"), ib=rand(heads), fb=rand(heads) + 2)
    S0, M0 = rand(nseq, heads, rows, N), rand(nseq, heads).abs()
    first = sum(lens[:seq])
    h, p = 1, P - 3

    def run():
        S, M, y, den = S0.clone(), M0.clone(), torch.empty(n, heads * P, device="cuda"), torch.ones(n, heads, device="cuda")
        _scan(form, heads, P, N, _portions(lens, [3] * nseq, list(range(nseq))), S, M, x, y, den)
        return S, M, y, den
    clean = run()
    x["xbc" if form == 0 else "proj"][first + j, h * P + p] = value
    S, M, y, den = run()
    col = h * P + p
    assert not torch.isfinite(y[first + j:first + lens[seq], col]).any()
    keep = torch.ones_like(y, dtype=torch.bool)
    keep[first + j:first + lens[seq], col] = False
    # (within the chunk of the token the products may be summed in another order: 16 of them, of the size of the largest outputs)
    assert torch.isfinite(y[keep]).all() and ((y - clean[2])[keep].abs() <= 16 * EPS * clean[2].abs().max()).all()
    hit = torch.zeros_like(S, dtype=torch.bool)
    hit[seq, h, p] = True
    assert not torch.isfinite(S[hit]).any() and torch.equal(S[~hit], clean[0][~hit])
    assert torch.equal(M, clean[1]) and torch.equal(den, clean[3])


@pytest.mark.parametrize("A_log,gates", [(100.0, (0.0, 0.0)), (80.0, (0.0, -3.0)), (30.0, (0.0, -40.0)), (5.0, (20.0, -8.0))],
                         ids=["overflows", "huge", "now and then", "large"])
@pytest.mark.parametrize("lens", [[37], [400]], ids=["whole", "segments"])
def test_decays_that_forget_everything(lens, A_log, gates):
    """A token may forget all before it (a decay of 0, or the rate itself overflows) between tokens that hardly forget anything."""
    heads, P, N, n = 1, 16, 64, sum(lens)
    g = torch.Generator(device="cuda").manual_seed(n)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    proj = torch.full((n, 8), gates[1], device="cuda")
    proj[::5] = gates[0]
    x = dict(xbc=rand(n, P + 2 * N), proj=proj, bias=torch.zeros(1, device="cuda"), A_log=torch.full((1,), A_log, device="cuda"), D=rand(1))
    S, y = rand(1, 1, P, N), torch.empty(n, P, device="cuda")
    st = S[0, 0].double()
    _scan(0, heads, P, N, _portions(lens, [1], [0]), S, None, x, y, None)
    xs, B, C = x["xbc"].double().split([P, N, N], 1)
    step = torch.nn.functional.softplus(proj[:, 0].double())
    a = torch.exp(-torch.exp(x["A_log"].double()) * step)
    # the rate and the step are 32-bit numbers of a few roundings each: a decay is off by that much of its exponent
    slack = (torch.exp(x["A_log"].double()) * step * a * 16 * EPS).nan_to_num(0.0)
    size, err = st.abs(), torch.zeros_like(st)
    for t in range(n):
        new = step[t] * xs[t][:, None] * B[t]
        err = a[t] * err + slack[t] * size
        st, size = a[t] * st + new, a[t] * size + new.abs()
        want, mag = st @ C[t] + x["D"].double() * xs[t], size @ C[t].abs() + (x["D"].double() * xs[t]).abs()
        assert ((y[t].double() - want).abs() <= (t + 1 + N + 32) * EPS * mag + err @ C[t].abs()).all(), t
    assert ((S[0, 0] - st).abs() <= (n + 32) * EPS * size + err).all()


@pytest.mark.parametrize("where", ["value", "key", "query"])
@pytest.mark.parametrize("huge", [-1e32, -3e38])
def test_silu_of_large_negative_inputs_is_nothing(where, huge):
    heads, P, N, n = 2, 64, 64, 40
    g = torch.Generator(device="cuda").manual_seed(7)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = dict(proj=rand(n, heads * (P + 2 * N)), rate=torch.full((heads,), 0.9, device="cuda"))
    S0 = rand(1, heads, P, N)
    col = {"value": 3, "key": heads * P + 5, "query": heads * (P + N) + 70}[where]

    def run(value):
        x["proj"][[4, 20, 39], col] = value
        S, y = S0.clone(), torch.empty(n, heads * P, device="cuda")
        _scan(1, heads, P, N, _portions([n], [1], [0]), S, None, x, y, None)
        return S, y
    for a, b in zip(run(huge), run(-200.0)):                    # (e^-200 is 0 in 32 bits)
        assert torch.equal(a, b)


@pytest.mark.parametrize("lens", [[17, 0, 17, 33] * 16, [16, 0, 33, 33, 1], [18, 20]], ids=["64", "ties", "two"])
@pytest.mark.parametrize("form,heads,P,N", [(0, 2, 64, 64), (1, 2, 16, 64), (2, 2, 24, 64)])
def test_portions_that_are_taken_by_length(form, heads, P, N, lens):
    """The longest first: equal lengths and portions without a token (of sequences that go on: their slots stay as they are) each find their own place."""
    test_chunked_recurrences_against_the_token_loop(form, heads, P, N, 1, lens, torch.bfloat16)


@pytest.mark.parametrize("lens,heads", [([50, 0, 17, 33] * 16, 5), ([60, 60, 1, 0] * 10, 7), ([70, 20], 130), ([1] * 63 + [48], 8)], ids=["64", "ties", "two", "one long"])
@pytest.mark.parametrize("form,P,N", [(0, 64, 64), (1, 16, 64), (2, 24, 64)])
def test_ragged_portions_in_more_workgroups_than_compute_units(form, P, N, lens, heads):
    """The same where the launch does take them by length: more than 256 workgroups, 48 tokens or more, lengths that differ."""
    assert heads * len(lens) > 256 and max(lens) >= 48 and 8 * sum(lens) <= 7 * max(lens) * len(lens)
    test_chunked_recurrences_against_the_token_loop(form, heads, P, N, 1, lens, torch.bfloat16)
