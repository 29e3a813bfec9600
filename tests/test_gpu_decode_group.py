"""GPU parity of the grouped decode kernel (several query heads per kv head)
at the sizes where it can go wrong: cache lengths around its 16-, 32- and
128-key rounds and one split, groups below, at and above the 16 columns of a
tile, head dims with idle V lanes, row strides, a running max that grows late.

Bound: K.Q has exact products and fp32 sums, P and V are not rounded, so an
fp32 output is within about S * 2^-24 of the weighted mean of |V|; 1e-5 holds
that for S < 5000 and |V| < 5.  16-bit outputs add one rounding."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(dev, B, H, Hkv, S, D, dtype, k_pad=0, boost=None):
    from minference.backend.attention import decode_dense

    g = torch.Generator("cpu").manual_seed(S + D + H)
    q = torch.randn(B, H, 1, D, generator=g).to(dtype)
    k, v = (torch.randn(B, S, Hkv, D + k_pad, generator=g).to(dtype) for _ in range(2))
    if boost:
        for j, f in boost:
            k[:, j] *= f
    qd, kd, vd = (t.to(dev) for t in (q, k, v))
    kv = [t[..., :D].transpose(1, 2) for t in (kd, vd)]
    out = torch.empty(q.shape, dtype=torch.float32, device=dev)
    decode_dense(qd, *kv, out=out)
    o16 = decode_dense(qd, *kv)
    qn = q.double().numpy()
    kn, vn = (t[..., :D].transpose(1, 2).double().numpy().repeat(H // Hkv, axis=1) for t in (k, v))
    x = (qn @ kn.swapaxes(-1, -2)) / np.sqrt(D)
    p = np.exp(x - x.max(-1, keepdims=True))
    ref = p @ vn / p.sum(-1, keepdims=True)
    assert np.abs(out.cpu().double().numpy() - ref).max() < 1e-5
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert (np.abs(o16.cpu().double().numpy() - ref) <= 1e-5 + ulp * np.abs(ref)).all()


@pytest.mark.parametrize("S", [1, 15, 16, 17, 31, 33, 64, 127, 128, 129, 500, 1025, 4113])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (96, torch.float16),
                                     (128, torch.bfloat16), (256, torch.float16)])
def test_lengths(gpu_device, S, D, dtype):
    _check(gpu_device, 2, 8, 2, S, D, dtype)


@pytest.mark.parametrize("H,Hkv", [(2, 1), (6, 2), (15, 1), (16, 1), (17, 1), (40, 1), (64, 2)])
def test_groups(gpu_device, H, Hkv):
    _check(gpu_device, 1, H, Hkv, 333, 96, torch.bfloat16)
    _check(gpu_device, 3, H, Hkv, 70, 512 if H < 10 else 128, torch.float16)


def test_row_stride_and_late_maximum(gpu_device):
    _check(gpu_device, 1, 4, 1, 900, 96, torch.bfloat16, k_pad=40)
    _check(gpu_device, 1, 4, 2, 2000, 128, torch.bfloat16,
           boost=[(3, 3.0), (700, 8.0), (1500, 30.0), (1999, 60.0)])


def _grouped_batch(H, S):
    """The smallest batch that the grouped kernel takes at every length and
    head dim: more than 512 64-key workgroups of one head each (smaller calls
    may go head by head)."""
    return 512 // (H * -(-S // 64)) + 1


@pytest.mark.parametrize("S", [1, 33, 129, 160, 257, 500, 1025])
@pytest.mark.parametrize("H,Hkv,D,dtype", [(8, 4, 64, torch.float16), (8, 2, 96, torch.bfloat16),
                                           (17, 1, 128, torch.bfloat16),
                                           (8, 2, 256, torch.float16), (4, 1, 512, torch.bfloat16)])
def test_lengths_of_many_heads(gpu_device, S, H, Hkv, D, dtype):
    _check(gpu_device, _grouped_batch(H, S), H, Hkv, S, D, dtype)


# Either side of every line between the kernels: 128 keys, 512 workgroups of a
# head, 16 MiB (24 at D = 512) read head by head.
@pytest.mark.parametrize("B,H,Hkv,S,D", [
    (1, 8, 4, 128, 128), (1, 8, 4, 129, 128), (1, 32, 8, 1024, 64), (1, 32, 8, 1025, 64),
    (1, 2, 1, 16383, 128), (1, 2, 1, 16384, 128), (1, 4, 1, 3071, 512), (1, 4, 1, 3072, 512),
    (1, 4, 1, 128, 512)])
def test_either_kernel(gpu_device, B, H, Hkv, S, D):
    _check(gpu_device, B, H, Hkv, S, D, torch.bfloat16)


# Rows past the cache's end: the last 16- or 32-key block of a wave reaches
# over S (by up to 31 rows), and those rows must read as zeros, whatever lies
# there.  The rows past S are NaN here, where 0 * NaN would show.  (2, 2): the
# kernel for one head per kv head, whose waves can be left without a block.
@pytest.mark.parametrize("H,Hkv", [(4, 1), (2, 2)])
@pytest.mark.parametrize("S", [1, 3, 15, 16, 17, 33, 64, 129, 1041])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (96, torch.float16),
                                     (128, torch.bfloat16), (256, torch.float16),
                                     (512, torch.bfloat16)])
def test_rows_past_the_cache_read_as_zeros(gpu_device, H, Hkv, S, D, dtype):
    from minference.backend.attention import decode_dense

    g = torch.Generator(gpu_device).manual_seed(S + D)
    B = _grouped_batch(H, S) if H > Hkv else 2
    q = torch.randn(B, H, 1, D, device=gpu_device, generator=g).to(dtype)
    k, v = (torch.randn(B, Hkv, S + 64, D, device=gpu_device, generator=g).to(dtype)
            for _ in range(2))
    k[:, :, S:], v[:, :, S:] = float("nan"), float("nan")
    ks, vs = k[:, :, :S], v[:, :, :S]
    out = decode_dense(q, ks, vs, out=torch.empty(q.shape, device=gpu_device))
    x = q.double() @ ks.double().repeat_interleave(H // Hkv, 1).transpose(-1, -2).contiguous()
    ref = torch.softmax(x / D ** 0.5, -1) @ vs.double().repeat_interleave(H // Hkv, 1)
    assert float((out - ref).abs().max()) < 1e-5  # the bound above


# Scores far below zero, down to the lowest finite ones: a row's softmax is of
# their differences, so the key with the smallest magnitude takes all of it.
# (2, 2): one head per kv head.
@pytest.mark.parametrize("H,Hkv", [(4, 1), (17, 1), (2, 2)])
@pytest.mark.parametrize("S", [1, 16, 33, 700])
@pytest.mark.parametrize("e", [55, 60, 62])  # scores about -2^(2e - 3), log2(1e30) is 99.7
def test_low_scores(gpu_device, H, Hkv, S, e):
    from minference.backend.attention import decode_dense

    D = 64
    g = torch.Generator(gpu_device).manual_seed(S)
    B = _grouped_batch(H, S) if H > Hkv else 1
    q = torch.zeros(B, H, 1, D, device=gpu_device, dtype=torch.bfloat16)
    k = torch.zeros(B, Hkv, S, D, device=gpu_device, dtype=torch.bfloat16)
    v = torch.randn(B, Hkv, S, D, device=gpu_device, generator=g).to(torch.bfloat16)
    q[..., 5] = 2.0 ** e
    k[..., 5] = -(2.0 ** e)
    top = (7 * S) // 11
    k[:, :, top, 5] = -(2.0 ** (e - 1))
    out = decode_dense(q, k, v, out=torch.empty(q.shape, device=gpu_device))
    want = v[:, :, top].float().repeat_interleave(H // Hkv, 1)
    assert torch.equal(out[:, :, 0], want)


@pytest.mark.parametrize("H", [4, 1])  # 1: one head per kv head
@pytest.mark.parametrize("S", [40, 300, 20000])
def test_infinite_scores(gpu_device, H, S):
    """-inf scores weigh nothing, wherever they stand; a row of nothing else
    gives 0; an infinite V stays in its own dim."""
    from minference.backend.attention import decode_dense

    D = 64
    g = torch.Generator(gpu_device).manual_seed(3)
    B = _grouped_batch(H, S) if H > 1 else 1
    q = torch.randn(B, H, 1, D, device=gpu_device, generator=g).to(torch.bfloat16)
    q[..., 0] = 1.0
    k, v = (torch.randn(B, 1, S, D, device=gpu_device, generator=g).to(torch.bfloat16)
            for _ in range(2))
    low = torch.arange(S, device=gpu_device) % 40 != 17  # whole 16- and 32-key blocks among them
    k[:, :, low, 0] = -float("inf")
    out = decode_dense(q, k, v, out=torch.empty(q.shape, device=gpu_device))
    x = q.double() @ k[:, :, ~low].double().transpose(-1, -2).contiguous() / D ** 0.5
    ref = torch.softmax(x, -1) @ v[:, :, ~low].double()
    assert float((out - ref).abs().max()) < 1e-5
    k[..., 0] = -float("inf")
    assert not decode_dense(q, k, v).any()
    # V: an infinite value reaches its own dim of every head and no other
    k = torch.randn(B, 1, S, D, device=gpu_device, generator=g).to(torch.bfloat16)
    v[:, 0, (7 * S) // 10, 9] = float("inf")
    out = decode_dense(q, k, v)
    assert torch.isinf(out[..., 9]).all()
    assert torch.isfinite(out[..., :9]).all() and torch.isfinite(out[..., 10:]).all()
