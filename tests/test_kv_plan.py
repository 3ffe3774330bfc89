"""The KV split by lengths on the CPU: its partial states fit the workspace that the page table's width sizes, its chunks
fit the grid, and chunks cover their sequences, whatever the lengths."""
import random

import pytest

import kv_plan


def _lens(rng, B, max_pages):
    top = max_pages * 16
    kind = rng.randrange(6)
    if kind == 0:
        return [top] * B
    if kind == 1:
        return [max(1, top * (i + 1) // B) for i in range(B)]
    if kind == 2:
        return [top] + [rng.randint(0, max(1, top // 16)) for _ in range(B - 1)]
    if kind == 3:
        lo = rng.uniform(0, 1)
        return [int(top * rng.uniform(lo, 1)) for _ in range(B)]
    if kind == 4:
        return [rng.choice([0, 1, top // 2, top - 1, top, top + 40]) for _ in range(B)]
    return [16 * rng.randint(0, max_pages) for _ in range(B)]


@pytest.mark.parametrize("ulps", [-1, 0, 1])
def test_states_and_chunks_fit(ulps):
    rng = random.Random(5 + ulps)
    ways = set()
    for _ in range(6000):
        B, hkv, group = rng.randint(1, 64), rng.choice([1, 2, 3, 4, 8, 16]), rng.choice([1, 5, 8, 16])
        max_pages = int(2 ** rng.uniform(0, 11.5))
        lens = _lens(rng, B, max_pages)
        f = kv_plan.fixed_plan(B, hkv, group, max_pages)
        s = kv_plan.split(lens, hkv, group, max_pages, ulps)
        ways.add((s.way, 2 * B > f.target))
        what = (lens, hkv, group, max_pages, s)
        assert s.states <= B * f.chunks, what
        assert sum(s.chunks) <= B * f.chunks + B and sum(s.chunks) < 1 << 15, what
        for n, c, per in zip(lens, s.chunks, s.per):
            assert c * per >= -(-min(n, 16 * max_pages) // 16), what
    assert {w for w, _ in ways} == {"fixed", "share", "half", "most", "last"}, ways


def test_sequences_that_fill_their_table_keep_the_plan_of_the_table():
    """Full tables up to the number of workgroups aimed at: the chunks of the table's own plan (17 chunks of 16 pages for
    one sequence of 264 pages, where an equal share that does not fit the states came out at 11 of 24)."""
    for B, hkv, max_pages in ((1, 8, 264), (1, 8, 2048), (4, 8, 256), (16, 8, 256), (16, 8, 2048), (64, 1, 128)):
        f = kv_plan.fixed_plan(B, hkv, 5, max_pages)
        for lens in ([16 * max_pages] * B, [16 * max_pages - 90] * B):
            s = kv_plan.split(lens, hkv, 5, max_pages)
            assert s.way == "fixed" and s.states == B * f.chunks, (B, hkv, max_pages, s)
    assert kv_plan.fixed_plan(1, 8, 5, 264).chunks == 17
