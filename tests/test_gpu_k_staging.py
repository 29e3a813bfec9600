"""Which calls stage K: the staged half of the workspace stays untouched where
the attention kernel reads K in place.  K is staged for a slow row stride (not
an odd multiple of 64 bytes) where the launch reads each tile often enough:
28 times at head dims below 128, 12 from 128 on; in a full prefill 8 times from
96 on (256: always between 257 and 512 items), at 64 30 times with 448 items or
more, else 60; always where the staging of a full prefill is told no heads."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _tensors(dev, H, Hkv, S_q, S_k, D, pad=0):
    q = torch.randn(1, H, S_q, D, device=dev).bfloat16()
    k = torch.randn(1, Hkv, S_k, D + pad, device=dev).bfloat16()[..., :D]
    v = torch.randn(1, Hkv, S_k, D, device=dev).bfloat16()
    return q, k, v


def _staged(k, ws):
    half = k.shape[0] * k.shape[1] * k.shape[3] * (-(-k.shape[2] // 64) * 64) * 2
    kt = ws[half:2 * half]
    return not bool((kt == 0x5A).all())


@pytest.mark.parametrize("H,Hkv,S_q,S_k,D,pad,staged", [
    (2, 2, 1000, 10000, 128, 0, True),     # 15 reads
    (2, 2, 1000, 10000, 64, 0, False),
    (2, 2, 2000, 10000, 64, 0, True),      # 29
    (2, 2, 700, 10000, 128, 0, False),     # 11
    (8, 2, 300, 10000, 128, 0, True),      # 20: 5 query blocks, groups of 4
    (2, 2, 2000, 10000, 64, 32, False),    # a fast stride
    (2, 2, 3700, 3700, 64, 0, False),      # full prefills: 29.5
    (2, 1, 3700, 3700, 64, 0, False),      # 59
    (2, 1, 3840, 3840, 64, 0, True),       # 61
    (8, 8, 3700, 3700, 64, 0, False),      # 464 items
    (8, 8, 3776, 3776, 64, 0, True),       # 30
    (4, 2, 3776, 3776, 64, 0, True),       # 60
    (2, 2, 896, 896, 96, 32, False),       # 7.5
    (2, 2, 960, 960, 96, 32, True),        # 8
    (2, 2, 960, 960, 128, 0, True),
    (2, 1, 448, 448, 128, 0, True),
    (2, 1, 300, 300, 128, 0, False),       # 6
    (2, 2, 960, 960, 256, 0, True),        # 8
    (2, 2, 896, 896, 256, 0, False),       # 7.5
    (18, 18, 896, 896, 256, 0, False),     # 252 items
    (19, 19, 896, 896, 256, 0, True),      # 266
    (37, 37, 896, 896, 256, 0, False),     # 518
    (2, 2, 300, 300, 512, 0, True),        # never read in place
])
def test_dense(gpu_device, H, Hkv, S_q, S_k, D, pad, staged):
    from minference import _abi

    q, k, v = _tensors(gpu_device, H, Hkv, S_q, S_k, D, pad)
    ws = _abi.workspace(_abi.attention_workspace_bytes(1, Hkv, S_k, D), gpu_device).fill_(0x5A)
    out = torch.empty_like(q)
    _abi.layer_attention(q, k, v, out, [(_abi.MSA_KIND_DENSE, 0, 0, -1, D ** -0.5)] * H, ws=ws)
    assert _staged(k, ws) == staged
    ref = torch.nn.functional.scaled_dot_product_attention(
        q.float().cpu(), k.float().cpu().repeat_interleave(H // Hkv, 1),
        v.float().cpu().repeat_interleave(H // Hkv, 1),
        attn_mask=torch.ones(S_q, S_k, dtype=torch.bool).tril(S_k - S_q))
    assert float((out.float().cpu() - ref).abs().max()) < 2e-2  # bf16 output below 4


@pytest.mark.parametrize("H,Hkv,S_q,S_k,D,staged", [
    (4, 4, 2000, 40000, 64, False),     # 32 query blocks of about 100 of 625 tiles: 5 reads
    (4, 4, 2000, 40000, 128, False),
    (16, 4, 2000, 20000, 128, True),    # 41
    (4, 4, 4000, 10000, 64, True),      # 40
    (4, 4, 700, 700, 64, True),
])
def test_sparse_layer(gpu_device, H, Hkv, S_q, S_k, D, staged):
    from minference import _abi

    q, k, v = _tensors(gpu_device, H, Hkv, S_q, S_k, D)
    ws = _abi.workspace(_abi.attention_workspace_bytes(1, Hkv, S_k, D), gpu_device).fill_(0x5A)
    est = _abi.workspace(_abi.estimate_workspace_bytes(1, 2, S_q, S_k, D), gpu_device)
    _abi.stage_kv_pool(q, k, v, [0, 1], est, ws)
    assert _staged(k, ws) == staged


def test_bands(gpu_device):
    """A band's reads do not grow with the length."""
    from minference import _abi

    q, k, v = _tensors(gpu_device, 2, 2, 6000, 6000, 128)
    n = _abi.attention_workspace_bytes(1, 2, 6000, 128)
    out = torch.empty_like(q)
    for n_local, staged in ((256, False), (1024, True)):  # 7 and 19 tiles with the sinks and the diagonal
        ws = _abi.workspace(n, gpu_device).fill_(0x5A)
        heads = [(_abi.MSA_KIND_STREAM, 64, n_local, -1, 128 ** -0.5)] * 2
        _abi.layer_attention(q, k, v, out, heads, ws=ws)
        assert _staged(k, ws) == staged
