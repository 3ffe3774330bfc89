"""The decode-GEMM's layout (tile height, shared tiles), restated from its rule (exl3_gemm.hip) for tests that name the code
they are for, and held to the library: a call without a workspace is refused with the size its own layout needs."""
from __future__ import annotations

import re
from dataclasses import dataclass

from trellis_serve_amd import _lib

CUS, COUNTERS, P = 256, 262144, 0x1000
SHAPES = ((4, 0.42, 20), (8, 0.62, 24), (12, 0.78, 32), (16, 0.95, 42))   # 16-row blocks, us per k-step, us of shared tiles


@dataclass
class Layout:
    height: int     # rows per tile
    tiles: int
    shared: int     # tiles cut into runs of k-steps over `groups` workgroups
    groups: int
    ksteps: int


def layout(rows: int, k: int, ns) -> Layout:
    nct, ksteps, best = sum((n // 128 + 1) // 2 for n in ns), k // 32, None
    for mi, step, shared_us in SHAPES:
        tiles = -(-rows // (16 * mi)) * nct
        rounds, rem = divmod(tiles, CUS)
        tile_us = ksteps * step + 8
        us, sk, groups = (rounds + (rem > 0)) * tile_us, 0, 0
        if rem:
            s = rem + CUS if rounds else rem
            g = max(1, min(CUS, s * ksteps // 8))
            shared = (tiles - s) // CUS * tile_us + s * ksteps / g * step + shared_us
            if shared < us:
                us, sk, groups = shared, s, g
        if best is None or us < best[0]:
            best = us, Layout(16 * mi, tiles, sk, groups, ksteps)
    out = best[1]
    lib = _lib.load()
    shards = (_lib.Exl3Shard * len(ns))(*[_lib.Exl3Shard(P, P, P, n) for n in ns])
    assert lib.exl3_linear_prefill(P, 0, rows, k, shards, len(ns), 3, 1, P, 0, P, 0, None) == _lib.EXL3_ERR_INVALID
    need = int(re.search(r"workspace 0 bytes, need (\d+)", lib.exl3_last_error().decode())[1])
    xh = (len(ns) * rows * k * 2 + 255) // 256 * 256
    assert need == COUNTERS + xh + out.groups * 2 * out.height * 1024, (out, need)
    return out
