"""msa_block_lists against its torch form: ids out of range, negative, far
beyond int32, repeated; one id and more ids than tiles; bitmaps of one word,
of a word's edge and of more than 64 words; all block sizes; int32 and int64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("block,s_q,s_k,topk", [
    (64, 1, 1, 1), (64, 64, 64, 3), (64, 65, 2048, 7), (64, 300, 2049, 65), (64, 130, 131073, 300),
    (128, 300, 300, 4), (192, 500, 1000, 5), (512, 700, 1500, 2), (64, 100, 1 << 20, 70)])
def test_lists(gpu_device, block, s_q, s_k, topk, dtype):
    from minference import _abi
    from minference.ops.block_sparse_kernel import canonical_block_lists, tile_ids

    n_bq, n_bk = -(-s_q // block), -(-s_k // block)
    g = torch.Generator().manual_seed(s_q + s_k)
    ids = torch.randint(-2, n_bk + 2, (2, 3, n_bq, topk), generator=g)
    ids[0, 0, 0, 0] = 2 ** 31 - 1
    if dtype == torch.int64:
        ids[0, 1, 0, 0], ids[1, 0, 0, 0] = 2 ** 62, -2 ** 62
    n_qt, n_kt = -(-s_q // 64), -(-s_k // 64)
    ref = ids.clamp(-1, n_bk + 1)  # the torch form multiplies the ids
    tiles = tile_ids(ref, block, n_qt) if block != 64 else ref
    want_idx, want_cnt = canonical_block_lists(tiles, n_kt)
    idx, cnt = _abi.block_lists(ids.to(dtype).to(gpu_device), block, s_q, s_k)
    assert torch.equal(cnt.cpu(), want_cnt) and torch.equal(idx.cpu(), want_idx)


def test_other_id_types(gpu_device):
    from minference.ops.block_sparse_kernel import block_sparse_attention_with_indices

    q, k, v = (torch.randn(1, 2, 300, 96, device=gpu_device).bfloat16() for _ in range(3))
    ids = torch.randint(0, 5, (1, 2, 5, 3))
    want = block_sparse_attention_with_indices(q, k, v, ids)
    for t in (ids.to(torch.int16), ids.to(torch.float32), ids.transpose(2, 3).contiguous().transpose(2, 3)):
        assert torch.equal(block_sparse_attention_with_indices(q, k, v, t), want)
    with pytest.raises(ValueError):
        block_sparse_attention_with_indices(q, k, v, ids[..., :0])


@pytest.mark.parametrize("block", [320, 1 << 20, (1 << 20) + 64, 1 << 33])
def test_block_beyond_the_keys(gpu_device, block):
    """One block that holds every token, at any size: id 0 is causal attention."""
    from minference.ops.block_sparse_kernel import block_sparse_attention_with_indices

    q, k, v = (torch.randn(1, 2, 300, 96, device=gpu_device).bfloat16() for _ in range(3))
    ids = torch.tensor([0, 1, -1, 0]).expand(1, 2, 1, 4)
    want = block_sparse_attention_with_indices(q, k, v, torch.arange(5).expand(1, 2, 5, 5))
    assert torch.equal(block_sparse_attention_with_indices(q, k, v, ids, block), want)
