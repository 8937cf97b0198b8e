"""The attention forward kernel where its key tiles go in halves to twice the waves: at the shortest lengths that take
that form, with a last tile whose second half is empty, one key long, or full, and with workgroups of which some
wave has no query."""
import pytest

import test_gpu_attention_parts as parts

pytestmark = pytest.mark.gpu

CASES = [(1, 4, 768), (1, 3, 769), (1, 2, 800), (1, 2, 801), (2, 1, 863), (1, 1, 1024), (1, 16, 1280), (1, 16, 1313),
         (1, 20, 1345)]


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("B,H,S", CASES)
def test_forward(hip, B, H, S, hd, causal):
    parts.test_forward(hip, B, H, S, hd, causal)
