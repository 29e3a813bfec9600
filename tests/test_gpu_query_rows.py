"""GPU parity of the query rows that the attention kernels load as whole rows:
one row and the edges of the 16 rows per wave and the 64 per block, rows
packed beside others, rows at both ends of their buffer, one row repeated
(row stride 0) and overlapping rows.

Bound: 2e-3 absolute on fp32 outputs, as for the other kernels (P rounded to
fp16: a row's error is at most 2^-11 of its weighted mean of |V|, |V| < 4)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from msa_data import make_qkv, np32

pytestmark = pytest.mark.gpu


def _views(q, layout):
    B, H, S, D = q.shape
    if layout == "packed":  # [S, H, 3 D] rows with something else beside them
        buf = torch.full((B, S, H, 3 * D), float("nan"), dtype=q.dtype, device=q.device)
        buf[..., D:2 * D] = q.transpose(1, 2)
        return buf[..., D:2 * D].transpose(1, 2)
    if layout == "repeated":
        return q[:, :, :1].contiguous().expand(B, H, S, D)
    if layout == "overlapping":  # row r starts 8 elements after row r - 1
        flat = torch.randn(B, H, D + 8 * S, generator=torch.Generator().manual_seed(S)).to(q)
        return flat.as_strided((B, H, S, D), (H * (D + 8 * S), D + 8 * S, 8, 1))
    return q


@pytest.mark.parametrize("D", [64, 96, 128, 256])
@pytest.mark.parametrize("layout", ["plain", "packed", "repeated", "overlapping"])
@pytest.mark.parametrize("S", [1, 15, 17, 49, 64, 65, 130])
def test_query_rows(gpu_device, D, layout, S):
    from minference import streaming_forward

    q, k, v = (t.to(gpu_device) for t in make_qkv(2, 2, S, S, D, torch.bfloat16, seed=S + D))
    q = _views(q, layout)
    out = torch.empty((2, 2, S, D), dtype=torch.float32, device=gpu_device)
    streaming_forward(q, k, v, 20, 90, out=out)
    ref, _ = O.layer_attention(np32(q), np32(k), np32(v), [("stream_llm", 20, 90)] * 2, "bf16")
    assert float(np.abs(out.cpu().numpy().astype(np.float64) - ref).max()) < 2e-3
