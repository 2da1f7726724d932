"""The gates of the real-gated recurrence on the 16-bit matrix instructions (csrc/seq/rglru_gates.hip) against 64 bits, and the scan that reads their pairs: matrices that
are bfloat16 numbers and such as need all three parts, rows that are no multiple of a wavefront's 32 or a pass's 256, inputs of very different size, an infinity."""
import pytest
import torch

from test_real_gated_recurrence_gpu import _portions

pytestmark = pytest.mark.gpu


def _case(n, blocks, exact, seed):
    g = torch.Generator().manual_seed(seed)
    u = (torch.randn(n, blocks * 128, generator=g) * torch.exp2(torch.randint(-6, 3, (n, blocks * 128), generator=g).float())).cuda()
    w = torch.randn(blocks, 128, 256, generator=g) * 128 ** -0.5
    w = (w.to(torch.bfloat16).float() if exact else w).cuda()
    b, lam = torch.randn(blocks, 1, 256, generator=g).cuda(), torch.rand(blocks * 128, generator=g).cuda()
    return u, w, b, lam


def _terms(u, w, b, lam, blocks):
    n = u.shape[0]
    z = torch.stack([u[:, k * 128:(k + 1) * 128].double() @ w[k].double() for k in range(blocks)]) + b.double()
    gr, gi = (z[:, :, s:s + 128].transpose(0, 1).reshape(n, -1) for s in (0, 128))
    la = -8.0 * torch.sigmoid(gr) * torch.nn.functional.softplus(lam.double())
    return la, torch.sqrt(-torch.expm1(2 * la)) * torch.sigmoid(gi) * u.double()


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("n,blocks", [(1, 3), (33, 1), (256, 2), (300, 130), (1500, 5)])
def test_pairs_against_64_bits(n, blocks, exact):
    from nano_vllm_amd import ops_seq
    u, w, b, lam = _case(n, blocks, exact, n)
    pairs = ops_seq.rglru_gates(u, w, b, lam, 8.0, blocks).double()
    for got, want in zip(pairs.unbind(-1), _terms(u, w, b, lam, blocks)):
        # sums of 128 products, each step 2^-24 of a sum of up to 20; a gate's slope is at most 1/4, and what follows costs a few units of the last place
        assert ((got - want).norm() / want.norm()).item() <= 5e-7


@pytest.mark.parametrize("lens", [[1] * 40, [700, 3, 90], [9]])
def test_scan_of_pairs_equals_the_scan_of_gates(lens):
    from nano_vllm_amd import ops_seq
    n, blocks = sum(lens), 4
    u, w, b, lam = _case(n, blocks, True, 7)
    ypre = torch.randn(n, 512, device="cuda")
    outs = []
    for ready in (True, False):
        S = torch.ones(len(lens), 512, device="cuda")
        out = torch.empty(n, 512, device="cuda")
        por = _portions(lens, [5] * len(lens))
        gates = ops_seq.rglru_gates(u, w, b, lam, 8.0, blocks) if ready else torch.baddbmm(b, u.view(n, blocks, 128).transpose(0, 1).contiguous(), w)
        ops_seq.rglru_scan(gates, None if ready else u, ypre, lam, 8.0, blocks, por, S, out)
        outs.append((out, S))
    for x, y in zip(*outs):
        # both are 32-bit sums of the same terms (2e-7 of each, above); decays below one do not add to that
        assert ((x - y).norm() / y.norm()).item() <= 1e-6


def test_an_infinite_input_stays_in_its_block():
    from nano_vllm_amd import ops_seq
    u, w, b, lam = _case(40, 2, True, 3)
    u[7, 5] = float("inf")
    pairs = ops_seq.rglru_gates(u, w, b, lam, 8.0, 2)
    z = u[:, :128].double() @ w[0].double() + b[0].double()
    assert torch.isfinite(pairs[:7]).all() and torch.isfinite(pairs[8:]).all() and torch.isfinite(pairs[7, 128:]).all()
    la = -8.0 * torch.sigmoid(z[7, :128]) * torch.nn.functional.softplus(lam[:128].double())       # gates of plus or minus infinity: 1 or 0
    assert torch.allclose(pairs[7, :128, 0].double(), la, rtol=1e-6, atol=1e-30)


@pytest.mark.parametrize("where", ["input", "matrix", "both"])
@pytest.mark.parametrize("exact", [True, False])
def test_infinities_beside_parts_that_are_zero(exact, where):
    """Weights whose second and third parts are 0 among such as need them, inputs of one part, an infinity in either: gates of plus or minus infinity are 1 or 0, and no
    other token or block is touched."""
    from nano_vllm_amd import ops_seq
    u, w, b, lam = _case(300, 2, exact, 5)
    w[0, 5, ::3] = 0.5
    w[0, 5, 1::3] = -1.0
    u[:, ::2] = u[:, ::2].bfloat16().float()
    calm = ops_seq.rglru_gates(u, w, b, lam, 8.0, 2)
    if where != "matrix":
        u[7, 5], u[270, 5] = float("inf"), -float("inf")
    if where != "input":
        w[0, 64, 70], w[0, 64, 200] = float("inf"), -float("inf")
    pairs = ops_seq.rglru_gates(u, w, b, lam, 8.0, 2)
    want = torch.stack(_terms(u, w, b, lam, 2), -1)
    lost = want.isnan().any(-1, keepdim=True)          # (infinities of both signs in one sum: a state that is multiplied by it is no number, whatever is added)
    assert torch.equal(pairs.isnan().any(-1, keepdim=True), lost) and torch.equal(pairs.isinf() & ~lost, want.isinf() & ~lost)
    finite = want.isfinite() & ~lost
    assert float((pairs.double() - want)[finite].norm() / want[finite].norm()) <= 5e-7
    touched = torch.zeros_like(finite)
    if where != "matrix":
        touched[[7, 270], :128] = True
    if where != "input":
        touched[:, [70, 200 - 128]] = True
    assert torch.equal(pairs[~touched], calm[~touched])
