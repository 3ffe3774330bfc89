"""Seeded random shapes through the fused linear (GEMV rows 1..16) and the prefill decode-GEMM (17..600 rows): k and
per-shard n of 128..5120 and 1..4 shards, every bit width and codebook, fp16 or bf16 input.  The split plans, shard
maps, tail tiles and half tiles take forms here that the fixed shapes of the other tests do not.  The reference is
built on the GPU from pieces pinned elsewhere -- the bit-exact reconstruct (W_inner), the input rotation of every
shard and an fp32 matmul, then the output rotation -- and the fused result must agree within the north-star
tolerance (norm-relative and max-relative 2e-3).  Outputs are fp16 (a bf16 input still gives an fp16 output)."""
import numpy as np
import pytest
import torch

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

# The decode-GEMM's tiles of 64, 128, 192 and 256 rows at their edges: one row, a row below, at and past each height,
# rows that leave a last tile of one row; whole tiles and shared runs of k-steps (a single k-step run included), shards
# that end in a half tile, every width of k-step data.  (K, codebook, k, ns, rows, bf16)
GEMM_EDGE_CASES = [(3, 1, 2048, (2176, 640), 1, False), (2, 0, 1280, (1024,), 63, False), (8, 2, 1280, (1024,), 64, True),
                   (4, 1, 512, (384, 128), 65, False), (5, 2, 1024, (4096,), 128, False),
                   (6, 0, 128, (128,), 129, False), (3, 1, 256, (17408, 17408), 192, False),
                   (3, 0, 256, (17408, 17408), 193, True), (4, 2, 640, (8192, 1152), 255, False),
                   (2, 1, 2048, (5120,), 257, False), (8, 0, 384, (896,), 385, False), (3, 1, 512, (16384,), 1025, False),
                   (5, 1, 5120, (8192, 1024), 700, False)]
# exl3_linear past 32 rows: large layers go to the decode-GEMM (from 4096 units of 128 x 128 weights), the last two
# stay on the GEMV
WIDE_LINEAR_CASES = [(3, 1, 8192, (8192,), 33, False), (4, 2, 5120, (6144, 6144, 1024), 48, True),
                     (2, 0, 17408, (5120,), 64, False), (3, 1, 8192, (8064,), 64, False), (3, 1, 8192, (8192,), 32, False)]


@pytest.mark.parametrize("case", GEMM_EDGE_CASES, ids=_ids(GEMM_EDGE_CASES))
def test_gemm_tile_heights_at_their_edges(case):
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
