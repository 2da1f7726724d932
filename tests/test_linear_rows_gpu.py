"""Linear layers of few rows (nvs_linear_rows) against float64: every tile the launcher chooses among, at the edges of its row and column
blocks, at reductions that give some wavefronts no piece or one fewer, on strided rows, with bias and with the activations."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(1, 16, 1), (1, 1, 3), (16, 1024, 8), (17, 30, 9), (32, 4100, 16), (33, 2050, 5), (64, 1024, 16), (64, 4096, 2), (65, 6144, 7), (100, 1030, 16),
         (129, 4096, 8), (256, 4090, 4), (256, 1024, 3)]              # rows, columns, pieces of 128 bytes of k


def case(dtype, m, n, pieces, glu, pad=0):
    g = torch.Generator(device="cuda").manual_seed(m * 10007 + n * 31 + pieces)
    k = pieces * (64 if dtype == torch.bfloat16 else 32)
    x = torch.randn(m, k + pad, generator=g, device="cuda").to(dtype)[:, :k]
    w = (torch.randn(n * (2 if glu else 1), k, generator=g, device="cuda") / k ** 0.5).to(dtype)
    b = torch.randn(n, generator=g, device="cuda").to(dtype)
    return x, w, b


def run(x, w, b, act, n, limit=0.0, alpha=0.0, pad=0):
    from nano_vllm_amd import ops_seq
    room = torch.full((x.shape[0], n + pad), 77.0, device="cuda", dtype=x.dtype)
    ops_seq._linear_rows(x, w, b, act, limit, alpha, room[:, :n])
    assert bool((room[:, n:] == 77.0).all()), "columns beyond the last were written"
    return room[:, :n].double()


def check(got, want, dtype, k):
    # an output is rounded once (8 bits in bf16: half of the last is up to 2^-8 of it; 2^-24 in 32-bit) from sums of k products in 32-bit: 4 sqrt(k) roundings of a sum's size
    size = want.abs().max()
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    assert bool(((got - want).abs() <= unit * want.abs() * 1.01 + 4 * k ** 0.5 * 2.0 ** -24 * size).all()), float((got - want).abs().max() / size)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,pieces", SIZES + [(330, 1024, 32), (330, 4096, 4), (512, 1540, 3), (1, 32770, 2)])
def test_products_and_bias(dtype, m, n, pieces):
    x, w, b = case(dtype, m, n, pieces, False, pad=16)
    want = x.double() @ w.double().T
    check(run(x, w, None, -1, n), want, dtype, x.shape[1])
    check(run(x, w, b, -1, n, pad=8), want + b.double(), dtype, x.shape[1])
    gelu = torch.nn.functional.gelu(want, approximate="tanh")
    check(run(x, w, None, 2, n), gelu, dtype, x.shape[1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,pieces", SIZES + [(330, 770, 16)])
def test_gated_activations(dtype, m, n, pieces):
    x, w, _ = case(dtype, m, n, pieces, True)
    z = x.double() @ w.double().T
    g, u = z[:, :n], z[:, n:]
    check(run(x, w, None, 0, n), torch.nn.functional.silu(g) * u, dtype, x.shape[1])
    g, u = g.clamp(max=1.25), u.clamp(-1.25, 1.25)
    check(run(x, w, None, 1, n, 1.25, 1.702, pad=3), g * torch.sigmoid(1.702 * g) * (u + 1), dtype, x.shape[1])


def test_the_layers_call_takes_every_size():
    """What the kernel does not cover goes to the library: short pieces, odd strides, many rows, other shapes."""
    from nano_vllm_amd import ops_seq
    for m, n, k, pad in ((0, 64, 64, 0), (3, 48, 40, 0), (5, 64, 64, 3), (5, 64, 64, 8), (600, 64, 64, 0), (40, 30000, 64, 0)):
        x = torch.randn(m, k + pad, device="cuda").bfloat16()[:, :k]
        w, b = torch.randn(n, k, device="cuda").bfloat16(), torch.randn(n, device="cuda").bfloat16()
        got, want = ops_seq.linear(x, w, b).double(), x.double() @ w.double().T + b.double()
        assert got.shape == want.shape and (m == 0 or float((got - want).abs().max()) <= 0.02 * float(want.abs().max()))
    with pytest.raises(RuntimeError):
        ops_seq.linear(torch.randn(3, 64, device="cuda"), torch.randn(64, 128, device="cuda"))
