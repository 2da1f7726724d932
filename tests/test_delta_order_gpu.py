"""The gated delta rule where portions are taken longest first, and where a head's columns go to two workgroups: every portion's rows and state are
those of the portion by itself, walked token by token."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,lens,d,dv,channelwise", [
    (37, [33, 0, 100, 33, 1, 16, 250, 7], 16, 24, True),          # by length: an empty portion, two of one length, a single token
    (129, [17, 40], 32, 16, False),                               # two portions, the second one longer
    (43, [20, 20, 20, 20, 20, 20], 16, 16, True),                 # all of one length
    (5, [(i * 37) % 50 + 1 for i in range(64)], 16, 16, False),   # as many as are taken by length
    (4, [(i * 23) % 40 + 1 for i in range(65)], 16, 16, True),    # one more: in their order
    (32, [40, 5, 90, 17], 128, 128, True),                        # 128 pairs: two workgroups of four wavefronts share a head's columns
])
def test_every_portion_is_as_by_itself(H, lens, d, dv, channelwise):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()
    n, ns = sum(lens), len(lens)
    starts = torch.tensor([0] + lens).cumsum(0).tolist()
    slots = torch.randperm(ns, generator=g).tolist()
    ctx = [3 * (i % 3) for i in range(ns)]
    qkv, gates = rnd(n, 2 * d + H * dv), rnd(n, 2 * H)
    decays = rnd(n, H * d) if channelwise else None
    A, dt = rnd(H) - 1.0, (rnd(H * d) if channelwise else rnd(H)) - 1.0
    S0 = 0.3 * rnd(ns, H, dv, d)

    def run(mode, group, S):
        part = slice(starts[group[0]], starts[group[-1] + 1])
        own = [lens[i] for i in group]
        cu = torch.tensor([0] + own).cumsum(0).int()
        seq = torch.repeat_interleave(torch.arange(len(own)), torch.tensor(own)).int()
        por = ops_seq.Portions(cu.cuda(), torch.tensor([ctx[i] for i in group]).int().cuda(), torch.tensor([slots[i] for i in group]).int().cuda(), seq.cuda(),
                               len(own), sum(own), max(own))
        y = torch.empty(por.n, H * dv, device="cuda")
        ops_seq.load_library().nvs_delta_force(mode)
        try:
            ops_seq.delta_scan(qkv[part].contiguous(), gates[part].contiguous(), H, 0, decays[part].contiguous() if channelwise else None, A, dt, d ** -0.5, H, 1, d, dv, por,
                               S, y)
        finally:
            ops_seq.load_library().nvs_delta_force(0)
        return y

    S1, S = S0.clone(), S0.clone()
    want = torch.cat([run(1, [i], S1) for i in range(ns) if lens[i]])
    got = run(2, list(range(ns)), S)
    # (32-bit sums in another order: 2e-5 of the largest, as the chunks' other tests allow)
    assert (got - want).abs().max() <= 2e-5 * want.abs().max()
    assert (S - S1).abs().max() <= 2e-5 * S1.abs().max()
