"""Products of many rows: what the kernels' offsets do not reach never gets to them. The callers' rule against csrc/seq/tiles_reach.h and the text of include/nvl_seq.h,
around the limits; on the GPU, calls at both sides of them."""
import os
import re
import shutil
import subprocess
from types import SimpleNamespace

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIMIT = (3 << 30) - 8192                        # bytes of an operand
SIZES = [(r, k, n * k, n) for r, k, n in [(393215, 4096, 4096), (393214, 4096, 4096), (393216, 4096, 256), (768, 4096, 393215), (768, 4096, 393214), (768, 128, 1 << 22),
                                          (768, 128, (1 << 22) - 8), (12582879, 128, 8), (12582880, 128, 8), (16384, 12288, 4096), (1, 128, 8)]]


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_callers_and_kernel_have_one_limit(tmp_path):
    from nano_vllm_amd import ops_seq
    calls = "\n".join(f'  std::printf("%d\\n", tiles_reach({r}ll, {ld}ll, {w}ll, {ldo}ll));' for r, ld, w, ldo in SIZES)
    src, exe = tmp_path / "reach.cpp", tmp_path / "reach"
    src.write_text('#include <cstdio>\n#include "tiles_reach.h"\nint main() {\n' + calls + "\n}\n")
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "nano_vllm_amd", "csrc", "seq"), str(src), "-o", str(exe)], check=True)
    told = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()
    with open(os.path.join(ROOT, "include", "nvl_seq.h")) as fh:
        said = re.search(r"n ldx and nout K below ([\d,]+) entries \(3 GiB less 8 KiB\), ldo below ([\d,]+)\.", fh.read())
    entries, ldo_limit = (int(s.replace(",", "")) for s in said.groups())
    assert entries * 2 == LIMIT
    for size, t in zip(SIZES, told):
        r, ld, w, ldo = size
        want = r * ld < entries and w < entries and ldo < ldo_limit
        assert ops_seq.tiles_reach(*size) == want == bool(int(t)), size


def test_gated_products_beyond_the_kernels_are_the_librarys():
    from nano_vllm_amd import ops_seq

    def stands_for(*shape):
        return SimpleNamespace(dtype=torch.bfloat16, is_cuda=True, device="cuda:0", shape=shape, dim=lambda: 2, stride=lambda i: (shape[1], 1)[i], is_contiguous=lambda: True,
                               numel=lambda: shape[0] * shape[1], data_ptr=lambda: 4096)
    w = stands_for(24576, 4096)
    assert ops_seq.silu_linear_fits(stands_for((8 << 20) - 256, 4096), w)
    assert not ops_seq.silu_linear_fits(stands_for((8 << 20) - 255, 4096), w)             # nvs_silu_linear: (n + 255) ldx < 2^35
    assert not ops_seq.silu_linear_fits(stands_for(1000, 4096), stands_for(8 << 20, 4096))


@pytest.mark.gpu
@torch.inference_mode()
@pytest.mark.parametrize("n,N,K,tiles", [(393214, 256, 4096, True), (393215, 256, 4096, False), (768, 393208, 4096, True), (768, 393216, 4096, False), (768, 1 << 22, 128, False)])
def test_layers_at_the_limits(n, N, K, tiles):
    """Operands between 2 and 3 GiB go through the tiles, whose offsets pass 2^31; what they do not reach is the library's, as before."""
    from nano_vllm_amd import ops_seq
    from nano_vllm_amd.layers import LinearBase
    ops_seq.load_library()
    x = torch.randn(n, K, dtype=torch.bfloat16, device="cuda")
    w = torch.randn(N, K, dtype=torch.bfloat16, device="cuda") / K ** 0.5
    assert ops_seq.tiles_rule(n, N, K) and ops_seq.many_rows(x, w) == tiles
    got = LinearBase.forward(SimpleNamespace(weight=w, bias=None, weight_packed=None), x)
    assert torch.equal(got, ops_seq.linear(x, w)) and got.shape == (n, N)
    for some in (slice(0, 300), slice(n // 2, n // 2 + 300), slice((1 << 31) // (2 * K) - 20, (1 << 31) // (2 * K) + 300), slice(n - 300, n)):
        for feats in (slice(0, 256), slice((1 << 31) // (2 * K) - 20, (1 << 31) // (2 * K) + 300), slice(N - 256, N)):
            want = x[some].double() @ w[feats].double().T
            if want.numel():              # bfloat16 has 8 significant bits: half a step is 2^-8 of a value at most; 4,096 sums in 32 bits around 1 stay below 2^-12
                assert ((got[some, feats].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -12).all()
