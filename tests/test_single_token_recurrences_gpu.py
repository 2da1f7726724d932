"""The matrix-state recurrences of single tokens (csrc/seq/scan_token.hip) against the token loop in float64: every size it is built for, fresh and continued sequences,
portions of no token between them, slots in any order."""
import pytest
import torch

from test_scan_chunks_gpu import test_chunked_recurrences_against_the_token_loop as against_the_token_loop

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("lens", [[1], [1, 0, 1, 1], [1] * 37], ids=["one", "gap", "crowd"])
@pytest.mark.parametrize("form,heads,G", [(0, 6, 2), (0, 3, 1), (1, 4, 1), (2, 4, 1)])
@pytest.mark.parametrize("P,N", [(32, 64), (64, 64), (128, 64), (32, 128), (64, 128), (128, 128)])
def test_single_tokens(form, heads, G, P, N, lens, dtype):
    against_the_token_loop(form, heads, P, N, G, lens, dtype)
