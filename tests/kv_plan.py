"""The split of a KV-attention batch over workgroups, restated from its rules for the tests (kv_attention.hip): the plan
by the page table's width, and the plan by the sequences' lengths that every wave derives, in float32 as on the device."""
from __future__ import annotations

from dataclasses import dataclass

import numpy as np

PAGE, CUS = 16, 256
F = np.float32


@dataclass
class Fixed:
    waves: int
    chunk_pages: int
    chunks: int
    target: int      # chunks per kv head aimed at


def fixed_plan(batch: int, hkv: int, group: int, max_pages: int) -> Fixed:
    waves = 4 if 8 * group * 131 * 4 > 65536 else 8
    aim = CUS if waves == 8 else 1024
    chunks = max(1, min(-(-max_pages // waves), -(-aim // (batch * hkv))))
    cp = -(-max_pages // chunks)
    cp = -(-cp // waves) * waves
    return Fixed(waves, cp, -(-max_pages // cp), -(-aim // hkv))


def by_length(batch: int, hkv: int, group: int, max_pages: int) -> bool:
    """Whether the call reads the lengths (and merges) at all."""
    f = fixed_plan(batch, hkv, group, max_pages)
    return batch <= 64 and f.chunk_pages > f.waves and not (
        f.chunks == 1 and (max_pages <= 16 * f.waves or batch * hkv >= 512))


@dataclass
class Split:
    way: str           # "fixed", or how the chunk length by lengths was found: "share", "half", "most", "last"
    chunks: list       # chunks per sequence
    per: list          # pages per chunk of each sequence
    states: int        # partial states written per (kv head, query head)


def rcp(x, ulps: int = 0):
    r = F(1) / F(x)
    for _ in range(abs(ulps)):
        r = np.nextafter(r, F(np.inf) if ulps > 0 else F(0), dtype=F)
    return r


def split(lens, hkv: int, group: int, max_pages: int, ulps: int = 0) -> Split:
    """ulps: the error of the device's approximate reciprocal."""
    B = len(lens)
    f = fixed_plan(B, hkv, group, max_pages)
    pages = [max(0, -(-min(n, max_pages * PAGE) // PAGE)) for n in lens]
    fixed = Split("fixed", [f.chunks] * B, [f.chunk_pages] * B, B * f.chunks if f.chunks > 1 else 0)
    if not by_length(B, hkv, group, max_pages):
        return fixed
    w, target, slots = f.waves, f.target, B * f.chunks
    worth = F(0.87) if slots <= target else F(1.6) if 2 * B <= target else F(1.1)
    total, live = F(sum(pages)), sum(p > 0 for p in pages)
    inv_target, inv_slots = F(1) / F(target), F(1) / F(slots)
    longest = [F(min(p, f.chunk_pages)) * worth for p in pages]
    if not any(x > total * max(inv_target, inv_slots) for x in longest):
        return fixed

    def up(x):
        return (int(x) + w) // w * w

    def chunks_of(cp):
        return [int(np.ceil(F(p) * rcp(cp, ulps))) for p in pages]

    def states(c):
        return sum(x for x in c if x > 1)

    crowded = 2 * live > target

    def fits(c):
        return states(c) <= slots and (crowded or sum(c) <= target)

    share = up(float(total) * float(inv_target) - 0.5)
    way, cp = "share", share
    if not fits(chunks_of(share)):
        room = max(min(target, slots) - live, 1)

        def leaving(part):
            return up(total * rcp(F(part * live + room), ulps))

        half, most, last = ((share + share // 2, 2 * share, up(max(F(3) * total * inv_slots, F(2) * share)))
                            if crowded else (leaving(0.5), leaving(0.25), leaving(0.0)))
        way, cp = ("half", half) if fits(chunks_of(half)) else ("most", most) if fits(chunks_of(most)) else ("last", last)
    if w == 8 and slots <= target and not any(x > cp for x in longest) and any(p > f.chunk_pages for p in pages):
        return fixed
    c = chunks_of(cp)
    per = [p if n <= 1 else -(-(-(-p // n)) // w) * w for p, n in zip(pages, c)]
    return Split(way, c, per, states(c))
