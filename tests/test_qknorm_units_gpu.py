"""The fused q/k norm, rotation and K/V store where a 16-lane row takes two heads: step sizes around the rule, last workgroups that are half
full, tokens without a slot — against the same kernel on the step's parts, which take one head each (bit for bit)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn], ids=["bf16", "fp8"])
@pytest.mark.parametrize("n,hq,hkv", [(8192, 16, 8), (8193, 16, 8), (15000, 16, 1), (37450, 5, 1), (9001, 28, 2)])
def test_two_heads_per_row_equal_one(n, hq, hkv, cache):
    from nano_vllm_amd import ops
    torch.manual_seed(n)
    dev = dict(device="cuda")
    block, heads = 256, hq + 2 * hkv
    assert n * heads >= 262144
    blocks = n // block + 2
    qkv = torch.randn(n, heads * 128, **dev).bfloat16()
    pos = torch.randint(0, 600, (n,), **dev)
    qw, kw = torch.randn(128, **dev).bfloat16(), torch.randn(128, **dev).bfloat16()
    table = torch.randn(500, 128, **dev)                        # positions beyond it are clamped
    slots = torch.randperm(blocks * block, **dev)[:n].int()
    slots[[0, 15, 16, n - 1]] = -1

    def run(parts):
        q, k = torch.zeros(n, hq, 128, **dev).bfloat16(), torch.zeros(n, hkv, 128, **dev).bfloat16()
        kc = torch.zeros(blocks, hkv, block, 128, **dev).to(cache)
        vc = torch.zeros_like(kc)
        for lo in range(0, n, parts):
            hi = min(lo + parts, n)
            ops.qknorm_rope_kvstore(qkv[lo:hi], pos[lo:hi], qw, kw, 1e-6, table, slots[lo:hi], q[lo:hi], k[lo:hi], kc, vc, hq, hkv)
        return q, k, kc.view(torch.int8), vc.view(torch.int8)
    for name, a, b in zip("q k k_cache v_cache".split(), run(n), run(2048)):
        assert torch.equal(a, b), name
