"""Linear layers on CPU tensors: products of every number of rows are torch's, also where the GPU library is loaded and no GPU is there."""
import pytest
import torch


@pytest.mark.parametrize("rows", [1, 300, 900, 2000])
@pytest.mark.parametrize("N,K", [(1024, 1024), (512, 2048)])
def test_products_of_cpu_tensors(rows, N, K):
    from nano_vllm_amd import ops_seq
    from nano_vllm_amd.layers import MergedColumnParallelLinear, ReplicatedLinear
    ops_seq.load_library()
    x, w = torch.randn(rows, K).bfloat16(), torch.randn(N, K).bfloat16()
    with torch.inference_mode():
        assert torch.equal(ops_seq.linear(x, w), torch.nn.functional.linear(x, w))
        layer = ReplicatedLinear(K, N).bfloat16()
        layer.weight.data.copy_(w)
        assert torch.equal(layer(x), torch.nn.functional.linear(x, w))
        both = MergedColumnParallelLinear(K, [N // 2] * 2).bfloat16()
        both.weight.data.copy_(w)
        assert torch.equal(both(x), torch.nn.functional.linear(x, w))
