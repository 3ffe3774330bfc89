"""Which form of the MoE layer a call takes, and what workspace it needs, on the CPU (no launch)."""
import pytest

import moe_plan


@pytest.mark.parametrize("E,top_k,H,I,tokens,K,ways", [
    # wide experts, few of them: the GEMVs read the weights once and are 8-40 % faster (272 against 379 us at the first)
    (8, 2, 4096, 14336, 64, 3, ("P2",)), (8, 2, 4096, 14336, 80, 2, ("P2",)), (8, 2, 6144, 16384, 52, 3, ("P2",)),
    (16, 2, 4096, 6400, 104, 3, ("P2",)), (16, 4, 5120, 8192, 40, 2, ("P2",)),
    # from two passes on, and with many narrow experts, the GEMMs
    (8, 2, 4096, 14336, 128, 3, ("gemm64",)), (128, 8, 2048, 768, 152, 3, ("gemm64",)),
    (128, 8, 2048, 768, 256, 8, ("gemm64",)), (60, 4, 2048, 1408, 150, 2, ("gemm64",)),
    (128, 8, 2048, 768, 37, 3, ("P1",)), (128, 8, 2048, 768, 1, 3, ("slot",)),
])
def test_the_faster_form_is_chosen(E, top_k, H, I, tokens, K, ways):
    """Calls where one form was measured clearly faster, at the edges of the rule."""
    assert moe_plan.way(tokens, top_k, E, H, I, K, K) in ways
