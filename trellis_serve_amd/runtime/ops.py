"""Custom ops, one opaque op per layer kind, as in the reference (cuda/src/sglang_exl3/runtime/ops.py:1-137):
row-count dispatch, dtype handling and output allocation live inside the op so a tracing engine sees one node.

`torch.ops.exl3_mi355x.linear(x, trellis[], suh[], svh[], codebook)` -> y [..., sum n_s] in x's dtype.
Dispatch (the reference's `_linear`, runtime/ops.py:62-126, with MI355X switch points):
  rows < PREFILL_ROWS  -> fused decode-GEMV (exl3_linear, up to 64 rows per launch)
  rows >= PREFILL_ROWS -> fused decode-GEMM (exl3_linear_prefill)
PREFILL_ROWS is the row count from which the fused GEMM is faster on every 27B shape: it decodes the weights once for up
to 256 rows.  Below it exl3_linear itself gives 33-64 rows of a large layer to the GEMM (48 rows: gate/up 81.5 -> 55 us,
down 61 -> 53) and keeps the narrow ones on the GEMV (q/k/v 33.5 us at 48 rows against 36, o 30 against 30-38).
"""
from __future__ import annotations

import os

import torch

from .. import ops as _kernels

PREFILL_ROWS = int(os.environ.get("EXL3_MI355X_PREFILL_ROWS", "65"))

_lib = torch.library.Library("exl3_mi355x", "FRAGMENT")  # must stay alive at module scope


def _linear(x: torch.Tensor, trellis: list[torch.Tensor], suh: list[torch.Tensor], svh: list[torch.Tensor],
            codebook: int) -> torch.Tensor:
    if x.dtype not in (torch.float16, torch.bfloat16):   # an fp32 caller: explicit cast, as the reference does
        return _linear(x.to(torch.float16), trellis, suh, svh, codebook).to(x.dtype)
    rows = x.shape[0] if x.dim() == 2 else x.reshape(-1, x.shape[-1]).shape[0]
    fn = _kernels.linear_prefill if rows >= PREFILL_ROWS else _kernels.linear
    return fn(x, trellis, suh, svh, codebook)   # [..., sum n_s]


def _linear_fake(x, trellis, suh, svh, codebook):
    return x.new_empty((*x.shape[:-1], sum(t.shape[1] * 16 for t in trellis)))


_lib.define("linear(Tensor x, Tensor[] trellis, Tensor[] suh, Tensor[] svh, int codebook) -> Tensor")
_lib.impl("linear", _linear, "CUDA")
torch.library.register_fake("exl3_mi355x::linear", _linear_fake, lib=_lib)

linear = torch.ops.exl3_mi355x.linear
