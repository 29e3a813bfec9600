"""vertical_and_slash on the GPU where its kernels can go wrong.

Estimator (indices bit-exact against the oracle): fewer than 64 rows, ragged
last key blocks, every entry ambiguous (its dot product a midpoint of two
values of the dtype, so each is recomputed exactly), equal keys (the top-k
decided by index), quotients by sqrt(D) of every magnitude the rounding of
the dtype can see, and more keys than one pass of the top-k's output takes.
Tile lists: sequence ends around 64 keys, repeated, negative and
out-of-range slashes."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from msa_data import dtype_tag, make_qkv, np32
from test_gpu_kernels import assert_close_f32, to_dev

pytestmark = pytest.mark.gpu


def _check(dev, q, k, vsz, ssz):
    from minference.ops.vertical_slash_kernel import vertical_and_slash_estimate

    gv, gs = vertical_and_slash_estimate(*to_dev(dev, q, k), vsz, ssz)
    rv, rs = O.vs_estimate(np32(q), np32(k), vsz, ssz, dtype_tag(q.dtype))
    assert np.array_equal(gv.cpu().numpy(), rv) and np.array_equal(gs.cpu().numpy(), rs)


@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S", [1, 15, 17, 63, 65, 127, 200, 1031])
@pytest.mark.parametrize("data", ["normal", "midpoints", "equal", "wide"])
def test_estimator(gpu_device, D, dtype, S, data):
    q, k, _ = make_qkv(1, 2, S, S, D, dtype, seed=S + D)
    if data == "midpoints":  # 257 (bf16) or 2049 (fp16) plus small even numbers
        big = 256.0 if dtype == torch.bfloat16 else 2048.0
        g = torch.Generator().manual_seed(S)
        q = torch.ones_like(q)
        k = torch.zeros_like(k)
        k[..., 0], k[..., 1] = big, 1.0
        k[..., 2] = (2 * torch.randint(0, 20, k.shape[:-1], generator=g)).to(dtype)
    elif data == "equal":
        k = k[:, :, :1].expand(1, 2, S, D).contiguous()
    elif data == "wide":
        g = torch.Generator().manual_seed(S)
        q, k = (t * torch.exp2(torch.randint(-9, 2, t.shape[:-1] + (1,), generator=g).float())
                .to(dtype) for t in (q, k))
    _check(gpu_device, q, k, max(1, S // 3), max(1, S // 2))


@pytest.mark.parametrize("data", ["normal", "equal"])
@pytest.mark.parametrize("S", [65536, 65537, 70001])
def test_topk_past_64k(gpu_device, data, S):
    q, k, _ = make_qkv(1, 1, S, S, 64, torch.bfloat16, seed=S)
    if data == "equal":
        k = k[:, :, :1].expand(1, 1, S, 64).contiguous()
    _check(gpu_device, q, k, 1000, 66000 if S > 66000 else 6096)


@pytest.mark.parametrize("S", [1, 63, 64, 65, 127, 129, 257])
@pytest.mark.parametrize("lo,hi", [(0, 1), (0, 300), (-200, 20), (60, 70)])
def test_tile_lists(gpu_device, S, lo, hi):
    from minference.ops.vertical_slash_kernel import vertical_slash_sparse_attention

    g = np.random.default_rng(S + hi)
    q, k, v = make_qkv(1, 2, S, S, 64, torch.bfloat16, seed=S)
    vi = np.sort(g.integers(0, S, (1, 2, 5)))
    si = np.sort(g.integers(lo, hi, (1, 2, 9)))[..., ::-1].copy()
    ref = O.vertical_slash_from_indices(np32(q), np32(k), np32(v), vi, si)
    out = torch.empty(q.shape, dtype=torch.float32, device=gpu_device)
    vertical_slash_sparse_attention(*to_dev(gpu_device, q, k, v), torch.from_numpy(vi),
                                    torch.from_numpy(si), out=out)
    assert_close_f32(out, ref, what=f"S={S} slashes in [{lo}, {hi})")
