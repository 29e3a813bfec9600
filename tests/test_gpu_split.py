"""GPU parity of the split attention kernel (head dims 128 and 256) and of the
rule that picks K in place or staged, at the sizes where they can go wrong:
one row, tile edges, one tile and many, rows with no visible key, late row
maxima (the rare path with its exchanged maxima), row strides on both sides of
the rule, more (batch, head) pairs than one item list holds.

Bound: 2e-3 absolute on fp32 outputs, as for the other kernels (P rounded to
fp16: a row's error is at most 2^-11 of its weighted mean of |V|, |V| < 4)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from msa_data import dtype_tag, make_qkv, np32

pytestmark = pytest.mark.gpu

TOL = 2e-3
PATS = [("stream_llm", 100, 200), ("block_sparse", 3, 0), ("dense", 0, 0), ("stream_llm", 0, 64)]


def _layer(dev, q, k, v, S_k):
    from minference.modules.minference_forward import build_layer_plan, run_layer_attention

    H, D = q.shape[1], q.shape[3]
    plan = build_layer_plan({h: [*PATS[h % 4], 1.0] for h in range(H)}, H, D, S_k)
    out = torch.empty(q.shape, dtype=torch.float32, device=dev)
    run_layer_attention(q, k, v, plan, out)
    ref, _ = O.layer_attention(np32(q), np32(k), np32(v), [PATS[h % 4] for h in range(H)],
                               dtype_tag(q.dtype))
    return float(np.abs(out.cpu().numpy().astype(np.float64) - ref).max())


@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (128, torch.float16),
                                     (256, torch.bfloat16), (256, torch.float16)])
@pytest.mark.parametrize("S_q,S_k", [(1, 1), (1, 64), (63, 63), (64, 64), (65, 65), (2, 130),
                                     (128, 128), (129, 1000), (513, 513)])
def test_edges(gpu_device, D, dtype, S_q, S_k):
    q, k, v = (t.to(gpu_device) for t in make_qkv(2, 4, S_q, S_k, D, dtype, seed=S_q + D,
                                                  sink_scale=8.0))
    assert _layer(gpu_device, q, k[:, :2], v[:, :2], S_k) < TOL


@pytest.mark.parametrize("D", [128, 256])
@pytest.mark.parametrize("factor", [4.0, 12.0, 40.0])
def test_late_maxima(gpu_device, D, factor):
    q, k, v = make_qkv(1, 4, 1100, 1100, D, torch.bfloat16, seed=int(factor))
    k = k.float()
    for j in (3, 70, 600, 601, 777, 1050):
        k[:, :, j] *= factor
    q, k, v = (t.to(gpu_device) for t in (q, k.to(torch.bfloat16), v))
    assert _layer(gpu_device, q, k, v, 1100) < TOL


@pytest.mark.parametrize("D", [128, 256])
def test_no_visible_key_and_full(gpu_device, D):
    from minference import dense_attention, streaming_forward

    q, k, v = (t.to(gpu_device) for t in make_qkv(1, 2, 200, 200, D, torch.bfloat16, seed=D))
    out = torch.full(q.shape, 7.0, dtype=torch.float32, device=gpu_device)
    streaming_forward(q, k, v, 0, 0, out=out)  # nothing is visible
    assert float(out.abs().max()) == 0.0
    dense_attention(q, k[:, :, :70], v[:, :, :70], causal=False, out=out)
    ref = O.dense_causal(np32(q), np32(k)[:, :, :70], np32(v)[:, :, :70], causal=False)
    assert float(np.abs(out.cpu().numpy() - ref).max()) < TOL


@pytest.mark.parametrize("D", [64, 96, 128, 256])
@pytest.mark.parametrize("pad", [0, 32, 64, 8, 40])
def test_row_strides(gpu_device, D, pad):
    """Row strides of D + pad elements: odd multiples of 64 bytes (K in
    place), multiples of 128 and 16-byte multiples that are neither (staged)."""
    S = 300
    ts = make_qkv(1, 4, S, S, D, torch.bfloat16, seed=pad + D, sink_scale=8.0)
    wide = [torch.full((1, 4, S, D + pad), float("nan"), dtype=t.dtype, device=gpu_device)
            for t in ts]
    for w, t in zip(wide, ts):
        w[..., :D] = t.to(gpu_device)
    q, k, v = (w[..., :D] for w in wide)
    assert _layer(gpu_device, q, k, v, S) < TOL


def test_many_pairs_plain_order(gpu_device):
    """More (batch, head) pairs than one item list: the plain item order."""
    q, k, v = (t.to(gpu_device) for t in make_qkv(17, 8, 65, 65, 128, torch.bfloat16, seed=17))
    assert _layer(gpu_device, q, k, v, 65) < TOL


@pytest.mark.parametrize("D", [96, 128, 256])
@pytest.mark.parametrize("j", [0, 63, 150, 299])
def test_non_finite_keys_and_values(gpu_device, D, j):
    """A NaN key reaches the rows that see it and no other; an infinite V its
    own dim of them."""
    from minference.backend.attention import dense_attention

    g = torch.Generator().manual_seed(j + D)
    q, k, v = (torch.randn(1, 2, 300, D, generator=g).half() for _ in range(3))
    mask = torch.ones(300, 300, dtype=torch.bool).tril()
    ref = torch.nn.functional.scaled_dot_product_attention(q.float(), k.float(), v.float(),
                                                           attn_mask=mask)

    def run(k, v):
        out = torch.empty(q.shape, device=gpu_device)
        return dense_attention(*(t.to(gpu_device) for t in (q, k, v)), out=out).cpu()

    bad = k.clone()
    bad[:, :, j, 3] = float("nan")
    out = run(bad, v)
    assert torch.isnan(out[:, :, j:]).all()
    if j:
        assert float((out - ref)[:, :, :j].abs().max()) < TOL
    bad = v.clone()
    bad[:, :, j, 9] = float("inf")
    out = run(k, bad)
    assert (out[:, :, j:, 9] == float("inf")).all()
    out[..., 9] = ref[..., 9]
    assert float((out - ref).abs().max()) < 2 * TOL  # |V| < 6 here: 2^-11 of 6
