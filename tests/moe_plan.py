"""Which form of the MoE layer a call takes, read back from the library: a call without a workspace is refused before any
launch with the size that its plan needs, and the sorted expert GEMMs' size is a closed form (exl3_moe.hip)."""
from __future__ import annotations

import ctypes
import math
import re

from trellis_serve_amd import _lib

COUNTERS = 262144   # EXL3_WORKSPACE_COUNTER_BYTES


def _up(v: int) -> int:
    return (v + 255) // 256 * 256


def gemm_bytes(tokens: int, top_k: int, E: int, H: int, I: int) -> int:
    """The workspace of the sorted expert GEMMs (tiles counted at 64 slots)."""
    slots = tokens * top_k
    return (COUNTERS + _up(8 * slots) + _up(8) + _up(16 * (slots // 64 + min(E, slots))) + _up(2 * slots * H)
            + _up(4 * slots * H) + _up(2 * slots * I))


def plan_bytes(tokens: int, top_k: int, E: int, H: int, I: int, K_gu: int = 3, K_dn: int = 3) -> int:
    """What the call's own plan needs."""
    lib = _lib.load()
    w = _lib.Exl3MoeWeights(*[0x1000] * 9)
    P = 0x1000
    rc = lib.exl3_moe_forward(P, 0, tokens, H, P, P, top_k, E, I, ctypes.byref(w), K_gu, K_dn, 1, P, 0, P, 0, None)
    assert rc == _lib.EXL3_ERR_INVALID
    m = re.search(r"workspace 0 bytes, need (\d+)", lib.exl3_last_error().decode())
    assert m, lib.exl3_last_error()
    return int(m[1])


def way(tokens: int, top_k: int, E: int, H: int, I: int, K_gu: int = 3, K_dn: int = 3) -> str:
    """"slot" (one token), "P1" / "P2" / "P4" (expert GEMVs of 16, 32, 64 slots a pass), "gemm64" / "gemm128"."""
    slots = tokens * top_k
    mean = slots / min(E, slots)
    if plan_bytes(tokens, top_k, E, H, I, K_gu, K_dn) == gemm_bytes(tokens, top_k, E, H, I):
        return "gemm128" if mean >= 128 else "gemm64"
    if tokens == 1 and slots <= E:
        return "slot"
    high = mean + 2.5 * math.sqrt(mean)
    return "P1" if high <= 16 else "P2" if high <= 32 else "P4"
