"""Seeded random shapes through the fused linear (GEMV rows 1..16) and the prefill decode-GEMM (17..600 rows): k and
per-shard n of 128..5120 and 1..4 shards, every bit width and codebook, fp16 or bf16 input.  The split plans, shard
maps, tail tiles and half tiles take forms here that the fixed shapes of the other tests do not.  The reference is
built on the GPU from pieces pinned elsewhere -- the bit-exact reconstruct (W_inner), the input rotation of every
shard and an fp32 matmul, then the output rotation -- and the fused result must agree within the
tolerance (norm-relative and max-relative 2e-3).  Outputs are fp16 (a bf16 input still gives an fp16 output)."""
import numpy as np
import pytest
import torch

import gemm_plan

pytestmark = pytest.mark.gpu
TOL = 2e-3


def _cases(seed, count, rows_lo, rows_hi, k_hi, n_hi):
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        K = int(rng.choice([2, 3, 4, 5, 6, 8]))
        cb = int(rng.integers(0, 3))
        k = 128 * int(rng.integers(1, k_hi // 128 + 1))
        shards = int(rng.integers(1, 5))
        ns = [128 * int(rng.integers(1, n_hi // 128 + 1)) for _ in range(shards)]
        M = int(rng.integers(rows_lo, rows_hi + 1))
        bf = bool(rng.random() < 0.3)
        out.append((K, cb, k, tuple(ns), M, bf))
    return out


GEMV_CASES = _cases(2026, 24, 1, 16, 5120, 3072)
PREFILL_CASES = _cases(2027, 10, 17, 600, 2048, 2048)


def _ids(cases):
    return [f"K{K}-cb{cb}-k{k}-n{'+'.join(map(str, ns))}-M{M}{'-bf16' if bf else ''}" for K, cb, k, ns, M, bf in cases]


def _run(case, prefill):
    from trellis_serve_amd import ops
    K, cb, k, ns, M, bf = case
    g = torch.Generator(device="cpu").manual_seed(hash(case) & 0xFFFFFFFF)
    trs = [torch.randint(-32768, 32768, (k // 16, n // 16, 16 * K), dtype=torch.int16, generator=g).cuda() for n in ns]
    suhs = [(torch.randint(0, 2, (k,), generator=g) * 2 - 1).half().cuda() for _ in ns]
    svhs = [(torch.randint(0, 2, (n,), generator=g) * 2 - 1).half().cuda() for n in ns]
    x = (torch.randn((M, k), generator=g) * 0.5).cuda()
    x = x.bfloat16() if bf else x.half()
    out = torch.empty((M, sum(ns)), dtype=torch.float16, device="cuda")
    fn = ops.linear_prefill if prefill else ops.linear
    y = fn(x, trs, suhs, svhs, cb, out=out).float()
    ref = torch.empty((M, sum(ns)), dtype=torch.float16, device="cuda")
    col = 0
    for tr, suh, svh in zip(trs, suhs, svhs):
        xh = ops.had_in_group(x, suh)
        w = ops.reconstruct(tr, cb)
        ops.had_out_into((xh.float() @ w.float()).half(), svh, ref, col)
        col += w.shape[1]
    ref = ref.float()
    nrel = ((y - ref).norm() / ref.norm()).item()
    mrel = ((y - ref).abs().max() / ref.abs().max()).item()
    assert nrel <= TOL and mrel <= TOL, (case, nrel, mrel)


# Rows at the edges of 64-row blocks, shards that end in a half tile, every width of k-step data; most of them small enough
# for tiles of 64 rows.  (K, codebook, k, ns, rows, bf16)
GEMM_EDGE_CASES = [(3, 1, 2048, (2176, 640), 1, False), (2, 0, 1280, (1024,), 63, False), (8, 2, 1280, (1024,), 64, True),
                   (4, 1, 512, (384, 128), 65, False), (5, 2, 1024, (4096,), 128, False),
                   (6, 0, 128, (128,), 129, False), (3, 1, 256, (17408, 17408), 192, False),
                   (3, 0, 256, (17408, 17408), 193, True), (4, 2, 640, (8192, 1152), 255, False),
                   (2, 1, 2048, (5120,), 257, False), (8, 0, 384, (896,), 385, False), (3, 1, 512, (16384,), 1025, False),
                   (5, 1, 5120, (8192, 1024), 700, False)]
# The decode-GEMM's tiles by height: a last tile that is full, short of one row, or one row; whole tiles only, every tile
# shared out by runs of k-steps ("shared"), and rounds of whole tiles before the shared ones ("rounds").  (case, rows per
# tile, kind)
GEMM_HEIGHT_CASES = [((2, 1, 1280, (128,), 64, False), 64, "shared"), ((3, 0, 1280, (128,), 65, True), 64, "shared"),
                     ((4, 2, 128, (128,), 256, False), 64, "whole"),
                     ((3, 1, 5120, (17408, 17408), 65, False), 128, "shared"), ((8, 2, 17408, (5120,), 128, False), 128, "shared"),
                     ((2, 0, 5120, (6144, 1024, 1024), 333, True), 128, "shared"),
                     ((5, 1, 4096, (2944,), 513, False), 128, "shared"), ((6, 2, 2560, (3712,), 512, True), 128, "shared"),
                     ((4, 1, 128, (4224, 2944), 513, False), 128, "whole"), ((3, 0, 128, (5760, 384, 1920), 512, False), 128, "whole"),
                     ((3, 1, 2048, (9344, 16768), 640, False), 128, "rounds"),
                     ((4, 0, 1280, (128, 17792, 640), 769, False), 192, "shared"), ((3, 2, 5120, (4224,), 575, True), 192, "shared"),
                     ((8, 1, 128, (9344,), 769, False), 192, "whole"), ((2, 2, 128, (9088, 1664), 768, True), 192, "whole"),
                     ((5, 1, 2048, (16512, 17536), 769, False), 192, "rounds"),
                     ((6, 0, 128, (10880,), 1025, False), 256, "whole"), ((3, 1, 128, (4480, 6016, 128), 1024, True), 256, "whole"),
                     ((4, 2, 5120, (2432, 10368), 442, False), 256, "shared"),
                     ((2, 1, 1024, (15488, 17792), 1023, False), 256, "rounds")]
# exl3_linear past 32 rows: large layers go to the decode-GEMM (from 4096 units of 128 x 128 weights), the last two
# stay on the GEMV
WIDE_LINEAR_CASES = [(3, 1, 8192, (8192,), 33, False), (4, 2, 5120, (6144, 6144, 1024), 48, True),
                     (2, 0, 17408, (5120,), 64, False), (3, 1, 8192, (8064,), 64, False), (3, 1, 8192, (8192,), 32, False)]


@pytest.mark.parametrize("case", GEMM_EDGE_CASES, ids=_ids(GEMM_EDGE_CASES))
def test_gemm_tile_heights_at_their_edges(case):
    _run(case, prefill=True)


@pytest.mark.parametrize("case,height,kind", GEMM_HEIGHT_CASES, ids=[f"{h}-{kind}-{i}" for (_, h, kind), i in
                                                                    zip(GEMM_HEIGHT_CASES, _ids([c[0] for c in GEMM_HEIGHT_CASES]))])
def test_gemm_tiles_by_height(case, height, kind):
    L = gemm_plan.layout(case[4], case[2], case[3])
    assert L.height == height
    assert kind == ("whole" if not L.shared else "shared" if L.shared == L.tiles else "rounds"), L
    _run(case, prefill=True)


@pytest.mark.parametrize("case", WIDE_LINEAR_CASES, ids=_ids(WIDE_LINEAR_CASES))
def test_linear_past_32_rows(case):
    _run(case, prefill=False)


@pytest.mark.parametrize("case", GEMV_CASES, ids=_ids(GEMV_CASES))
def test_random_gemv_shapes(case):
    _run(case, prefill=False)


@pytest.mark.parametrize("case", PREFILL_CASES, ids=_ids(PREFILL_CASES))
def test_random_prefill_shapes(case):
    _run(case, prefill=True)
