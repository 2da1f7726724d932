"""The centered norm of one group whose row stays in registers, at the edges of the accesses per thread (4 columns x 1, 2, 4, 8)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [4, 1020, 1024, 1028, 2048, 2052, 4096, 4100, 8192, 8196])
def test_centered_rows(W):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(W)
    n, eps = 5, 1e-3
    x0, a, b = torch.randn(n, W, generator=g) + 20, torch.randn(n, W, generator=g), torch.randn(n, W, generator=g)
    w = 1 + torch.randn(W, generator=g)
    x, out = x0.cuda(), torch.empty(n, W, device="cuda")
    ops_seq.add_group_norm(x, w.cuda(), 1, eps, out, a=a.cuda(), b=b.cuda(), a_mult=0.5, center=True)
    s = x0.double() + 0.5 * a.double() + b.double()
    assert ((x.cpu().double() - s).abs() <= 3 * 2.0 ** -24 * (s.abs() + a.abs() + b.abs())).all()
    want = torch.nn.functional.layer_norm(s, (W,), w.double(), None, eps)
    # an entry is (s - mean) k w: s carries 3 roundings of about 20, the mean those of a sum in log2(W) + 8 stages, k a handful
    scale = (s.var(1, unbiased=False, keepdim=True) + eps).rsqrt()
    stages = 8 + W.bit_length()
    tol = 2.0 ** -24 * w.abs() * (scale * 25 * (3 + stages) + (stages + 6) * want.abs() / w.abs().clamp(min=1e-9))
    assert ((out.cpu().double() - want).abs() <= tol).all()
