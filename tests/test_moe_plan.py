"""Which form of the MoE layer a call takes, and what workspace it needs, on the CPU (no launch)."""
import pytest

import moe_plan
from trellis_serve_amd import _lib


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


@pytest.mark.parametrize("E,top_k,H,I,K_gu,K_dn", [
    (8, 2, 4096, 14336, 3, 3), (60, 4, 2048, 1408, 3, 3), (128, 8, 2048, 768, 3, 4), (128, 8, 2048, 768, 8, 2),
    (16, 6, 1024, 512, 2, 2), (8, 1, 128, 128, 3, 3), (1, 1, 16384, 128, 5, 5), (1, 1, 128, 2048, 2, 8), (256, 8, 1280, 768, 4, 4),
    (2, 2, 7168, 2048, 6, 6), (512, 3, 2048, 512, 2, 3), (64, 64, 1024, 1024, 3, 3)])
def test_workspace_of_the_most_tokens_serves_fewer(E, top_k, H, I, K_gu, K_dn):
    """A workspace sized for a caller's most tokens serves every smaller call (as a call's own plan states its need)."""
    lib = _lib.load()
    most = min(4096, ((1 << 29) - 1) // (top_k * max(2 * I, H)))
    reported = worst = 0
    ways = set()
    for t in range(1, most + 1):
        if t > 600 and t % 37:
            continue
        size = lib.exl3_moe_workspace_bytes(t, top_k, E, H, I, K_gu, K_dn)
        assert size >= reported, t
        reported = size
        worst = max(worst, moe_plan.plan_bytes(t, top_k, E, H, I, K_gu, K_dn))
        assert size >= worst, t
        ways.add(moe_plan.way(t, top_k, E, H, I, K_gu, K_dn)[:4])
    if E <= 256 and 1024 <= H <= 4096 and top_k <= 8:
        assert {"gemm"} < ways
