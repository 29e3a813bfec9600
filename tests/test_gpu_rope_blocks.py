"""The fused RoPE at token counts around the lines between its block sizes
(1, 4 and 16 tokens) and their remainders, bit-exact with the eager form."""

from __future__ import annotations

import pytest
import torch

from test_rope import hf_rope

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S", [(1, 3), (1, 511), (1, 512), (1, 515), (3, 171), (2, 1023), (1, 3071),
                                 (1, 3072), (1, 3085), (3, 1029)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_token_counts(gpu_device, B, S, dtype):
    from minference.ops.rope import apply_rotary_pos_emb

    g = torch.Generator(gpu_device).manual_seed(S)
    qkv = torch.randn(B, S, (6 + 4) * 96, device=gpu_device, generator=g).to(dtype)
    q = qkv[..., :6 * 96].view(B, S, 6, 96).transpose(1, 2)
    k = qkv[..., 6 * 96:8 * 96].view(B, S, 2, 96).transpose(1, 2)
    cos, sin = (torch.randn(B, S, 96, device=gpu_device, generator=g).to(dtype) for _ in range(2))
    want = hf_rope(q, k, cos, sin)
    got = apply_rotary_pos_emb(q, k, cos, sin)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
