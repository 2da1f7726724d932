"""Products of 257 to 1,024 rows on the few-row kernel: results at the edges of its tiles, and whose products they stay."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,N,K,bias,pad", [(257, 8, 64, False, 0), (320, 1040, 1024, True, 0), (1000, 1024, 2048, False, 8), (1024, 1024, 64, True, 64), (512, 2048, 128, True, 0),
                                            (383, 3072, 1024, False, 0), (449, 4096, 1024, True, 0), (770, 100, 192, True, 8)])
def test_results_at_the_edges(m, N, K, bias, pad):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, K + pad, generator=g).bfloat16().cuda()[:, :K]
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    b = torch.randn(N, generator=g).bfloat16().cuda() if bias else None
    with torch.inference_mode():
        assert ops_seq.some_rows(x, w, b)
        got = ops_seq.linear(x, w, b).double()
    want = x.double() @ w.double().t() + (b.double() if bias else 0.0)
    # rounding to 16 bits, half a unit of 8 bits, and K sums in 32 bits of products up to the sum of their sizes
    bound = want.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().t()) * K * 2.0 ** -24 + 1e-30
    assert bool(((got - want).abs() <= bound).all())


def test_products_that_stay_the_library_s():
    from nano_vllm_amd import ops_seq
    ops_seq.load_library()
    x, w = torch.randn(300, 128, device="cuda").bfloat16(), torch.randn(64, 128, device="cuda").bfloat16()
    with torch.no_grad():
        assert ops_seq.some_rows(x, w)
        assert not ops_seq.some_rows(x.t().contiguous().t(), w) and not ops_seq.some_rows(x[:, 4:], w[:, :124].contiguous()) and not ops_seq.some_rows(x.float(), w.float())
        assert not ops_seq.some_rows(x.expand(2, 300, 128), w) and not ops_seq.some_rows(x[:1].expand(300, 128), w)
        with torch.autocast("cuda", dtype=torch.float16):
            assert not ops_seq.some_rows(x, w)

        class Mine(torch.Tensor):
            pass
        assert not ops_seq.some_rows(x.as_subclass(Mine), w)
    w.requires_grad_(True)
    assert not ops_seq.some_rows(x, w)
    y = ops_seq.linear(x, w)
    y.sum().backward()
    assert w.grad is not None


def test_a_captured_product_of_two_passes_is_the_library_s_and_one_of_one_pass_is_not():
    from nano_vllm_amd import ops_seq
    assert ops_seq.rows_rule(400, 4096, 1024) and not ops_seq.rows_rule(400, 4096, 1024, captured=True) and not ops_seq.rows_rule(400, 4096, 2048)
    assert ops_seq.rows_rule(1000, 1024, 4096, captured=True) and not ops_seq.rows_rule(1025, 1024, 4096) and not ops_seq.rows_rule(770, 1040, 2048)
    assert not ops_seq.rows_rule(64, 12288, 4096) and not ops_seq.rows_rule(256, 4096, 4096) and ops_seq.rows_rule(257, 2048, 4096)
    x, w = torch.randn(400, 1024, device="cuda").bfloat16(), torch.randn(1024, 1024, device="cuda").bfloat16()
    with torch.inference_mode():
        want = ops_seq.linear(x, w)
        s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            got = ops_seq.linear(x, w)
        for _ in range(3):
            got.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want)


def test_which_steps_wait_for_the_host():
    """Prompt steps behind short contexts do, by what they say of themselves; those behind long ones, decode steps and captured ones do not, and their products stay the library's."""
    from types import SimpleNamespace

    from nano_vllm_amd import ops_seq
    from nano_vllm_amd.attn_meta import reset_context, set_context
    ops_seq.load_library()
    x, w = torch.randn(320, 1024, device="cuda").bfloat16(), torch.randn(4096, 1024, device="cuda").bfloat16()
    cu = torch.tensor([0, 320], dtype=torch.int32, device="cuda")
    steps = [(True, (True, cu, cu, 320, 320), {}), (True, (True, cu, cu, 320, 2304), {}), (False, (True, cu, cu, 320, 2305), {}), (False, (False,), dict(context_lens=cu)),
             (True, (False,), {}), (True, (True,), dict(portions=SimpleNamespace(max_q=2))), (False, (True,), dict(portions=SimpleNamespace(max_q=1)))]
    try:
        with torch.inference_mode():
            for waits, args, kw in steps:
                set_context(*args, **kw)
                assert ops_seq.waits_for_host() == waits and ops_seq.some_rows(x, w) == waits and ops_seq.silu_short_steps(320, 1024) == waits, (args, kw)
                assert ops_seq.some_rows(x, w[:1024])                  # one pass: in every step
                assert not ops_seq.silu_short_steps(320, 1088) and not ops_seq.silu_short_steps(63, 1024)
    finally:
        reset_context()
