"""Row kernels of four columns (or 16 bytes) per access, with rows in registers: widths at the edges of the accesses per thread and just off the
vector path, against the definitions in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def _rms(v, eps=1e-5):
    return v / torch.sqrt(v.pow(2).mean(-1, keepdim=True) + eps)


@pytest.mark.parametrize("W", [4, 254, 1020, 1028, 2048, 4100, 8192, 8196])
@pytest.mark.parametrize("two", [False, True])
def test_norm_and_residual(W, two):
    from nano_vllm_amd import ops_seq
    torch.manual_seed(W)
    n = 3
    m, m2, x0 = (torch.randn(n, W, device="cuda") for _ in range(3))
    w1, w2, g = torch.randn(W, device="cuda"), torch.randn(W, device="cuda"), torch.tensor([0.7], device="cuda")
    x, xh = x0.clone(), torch.empty_like(x0)
    ops_seq.norm_residual(x, m, g, 1e-5, xh, *((m2, w1, w2) if two else ()))
    v = _rms(m.double())
    if two:
        v = _rms(0.5 * (v * w1.double() + _rms(m2.double()) * w2.double()))
        size = _rms(m.double()).abs() * w1.double().abs() + _rms(m2.double()).abs() * w2.double().abs()
        size = size / torch.sqrt((0.5 * (_rms(m.double()) * w1.double() + _rms(m2.double()) * w2.double())).pow(2).mean(-1, keepdim=True) + 1e-5)
    else:
        size = v.abs()
    want = x0.double() + g.double() * v
    # a root mean square is a sum of log2(W) + 8 stages; a dozen roundings around it
    tol = EPS * (want.abs() + (W.bit_length() + 20) * size)
    assert ((x.double() - want).abs() <= tol).all() and torch.equal(x, xh)


@pytest.mark.parametrize("group", [512, 516, 1020, 1024, 1028, 2052, 4096, 8192, 8196])
@pytest.mark.parametrize("order", ["gate first", "norm first", "silu"])
def test_gate_and_wide_groups(group, order):
    from nano_vllm_amd import ops_seq
    torch.manual_seed(group)
    n, groups = 3, 2
    W = group * groups
    y, z, w = torch.randn(n, W, device="cuda"), torch.randn(n, W + 8, device="cuda")[:, 4:4 + W], torch.randn(W, device="cuda")
    out = torch.empty(n, W, device="cuda")
    ops_seq.gated_group_norm(y, z, w, groups, 1e-5, out, norm_first=order != "gate first", silu=order == "silu")
    zd, yd = z.double(), y.double()
    gate = torch.sigmoid(zd) if order == "norm first" else torch.nn.functional.silu(zd)
    if order == "gate first":
        want = _rms((yd * gate).view(n, groups, group)).reshape(n, W) * w.double()
    else:
        want = _rms(yd.view(n, groups, group)).reshape(n, W) * w.double() * gate
    assert ((out.double() - want).abs() <= (group.bit_length() + 24) * EPS * want.abs() + 1e-12).all()


@pytest.mark.parametrize("shape,dtype", [((3, 5), torch.float32), ((7, 4), torch.float32), ((1, 2056), torch.bfloat16), ((13, 1001), torch.bfloat16),
                                         ((48, 4096), torch.float32), ((96, 2048), torch.bfloat16), ((201, 1000), torch.bfloat16), ((49, 4095), torch.float32)])
@pytest.mark.parametrize("scale", [0.01, 1.0, 30.0])
def test_xielu(shape, dtype, scale):
    from nano_vllm_amd import ops_seq
    torch.manual_seed(shape[1])
    z = (torch.randn(shape, device="cuda") * scale).to(dtype)
    pq = torch.tensor([0.4, -0.3], device="cuda", dtype=dtype)
    zd = z.double()
    ap, aq = torch.nn.functional.softplus(pq.double())
    aq = aq + 0.5
    curve = torch.where(zd > 0, ap * zd * zd, aq * (torch.expm1(zd) - zd))
    got = ops_seq.xielu(z.clone(), pq).double()
    size = curve.abs() + 0.5 * zd.abs()
    assert ((got - (curve + 0.5 * zd)).abs() <= (8 * EPS + (2.0 ** -8 if dtype == torch.bfloat16 else 0)) * size).all()


@pytest.mark.parametrize("W", [4, 6, 1020, 1028, 4096])
def test_rows_with_a_sinusoid(W):
    from nano_vllm_amd import ops_seq
    torch.manual_seed(W)
    n, table = 5, torch.randn(11, W, device="cuda")
    ids, pos = torch.randint(0, 11, (n,), device="cuda"), torch.tensor([0, 1, 7, 100, 500], device="cuda")
    x, xh = torch.empty(n, W, device="cuda"), torch.empty(n, W, device="cuda")
    ops_seq.embed_sinusoid(table, ids, pos, 1.5, 10000.0, x, xh)
    i = (torch.arange(W, device="cuda") // 2).double()
    angle = pos.double()[:, None] * 10000.0 ** (-2 * i / W)
    want = table[ids].double() * 1.5 + torch.where(torch.arange(W, device="cuda") % 2 == 1, angle.cos(), angle.sin())
    # the frequency is a 32-bit power of two of an exponent of up to 13.3: a few 1e-6 of the angle
    assert ((x.double() - want).abs() <= 4e-6 * angle + 1e-6).all() and torch.equal(x, xh)
