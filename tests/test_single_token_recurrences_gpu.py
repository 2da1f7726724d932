"""The matrix-state recurrences of single tokens (csrc/seq/scan_token.hip) against the token loop in float64: every size it is built for, fresh and continued sequences,
portions of no token between them, slots in any order."""
import pytest
import torch

import test_scan_chunks_gpu
from test_scan_chunks_gpu import test_chunked_recurrences_against_the_token_loop as against_the_token_loop

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("lens", [[1], [1, 0, 1, 1], [1] * 37], ids=["one", "gap", "crowd"])
@pytest.mark.parametrize("form,heads,G", [(0, 6, 2), (0, 3, 1), (1, 4, 1), (2, 4, 1)])
@pytest.mark.parametrize("P,N", [(32, 64), (64, 64), (128, 64), (32, 128), (64, 128), (128, 128)])
def test_single_tokens(form, heads, G, P, N, lens, dtype):
    against_the_token_loop(form, heads, P, N, G, lens, dtype)


@pytest.mark.parametrize("form,heads,G,P,N", [(0, 6, 2, 64, 128), (1, 4, 1, 128, 128), (2, 4, 1, 32, 64), (2, 2, 1, 128, 128)])
def test_portions_longer_than_the_caller_said(form, heads, G, P, N, monkeypatch):
    """The longest portion chooses the kernel; one that is too small costs time, not results."""
    def as_single_tokens(lens, ctx, slots, plain=test_scan_chunks_gpu._portions):
        p = plain(lens, ctx, slots)
        p.max_q = 1
        return p
    monkeypatch.setattr(test_scan_chunks_gpu, "_portions", as_single_tokens)
    against_the_token_loop(form, heads, P, N, G, [2, 5, 1, 0, 3], torch.float32)
