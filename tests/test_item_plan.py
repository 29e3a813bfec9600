"""What the key splits of a launch ask for (msa_split_workspace_bytes, host
arithmetic): nothing where the whole items fill the GPU's rounds, and each long
head's own number of pieces elsewhere."""

from __future__ import annotations

import ctypes

import pytest

from minference import _abi

DENSE, STREAM, BLOCK = _abi.MSA_KIND_DENSE, _abi.MSA_KIND_STREAM, _abi.MSA_KIND_BLOCK


def split_groups(heads, S_q, S_k, Hkv, D):
    """Partial outputs (key splits of all split heads) of one launch."""
    H = len(heads)
    t = [_abi.MsaTensor4() for _ in range(2)]
    for d, n, s in zip(t, (H, Hkv), (S_q, S_k)):
        d.data = 0x10000
        d.size[:] = [1, n, s, D]
        d.stride[:] = [n * s * D, s * D, D, 1]
        d.dtype = _abi.MSA_DTYPE_BF16
    arr = _abi.head_descs([(kind, p1, p2, 0, 0.1) for kind, p1, p2 in heads])
    n = _abi.load_library().msa_split_workspace_bytes(ctypes.byref(t[0]), ctypes.byref(t[1]), arr, H,
                                                      100)
    per = -(-S_q // 64) * 64 * (D + 2) * 4
    assert n % per == 0
    return n // per


@pytest.mark.parametrize("D", [64, 96, 128])
@pytest.mark.parametrize("S_k", [10000, 20000, 40000])
def test_full_rounds_stay_whole(D, S_k):
    """512 items of one length are one round of the 512 workgroups."""
    assert split_groups([(DENSE, 0, 0)] * 32, 1000, S_k, 32, D) == 0
    assert split_groups([(BLOCK, 100, 0), (STREAM, 128, 4096)] * 16, 1000, S_k, 8, D) == 0


def test_pieces_follow_each_head():
    """100 rows of 40000 keys: 625-tile heads in 8, 100-tile heads in 4 and
    68-tile heads in 3 pieces of at most 32 tiles at D = 128; below it pieces
    have up to 64 tiles, the 68-tile heads stay whole, and the 100-tile heads
    too once the items outnumber the CUs."""
    heads = [(DENSE, 0, 0)] * 3 + [(BLOCK, 100, 0)] * 19 + [(STREAM, 128, 4096)] * 10
    assert split_groups(heads, 100, 40000, 8, 128) == 3 * 8 + 19 * 4 + 10 * 3
    assert split_groups(heads, 100, 40000, 8, 96) == 3 * 8 + 19 * 2
    assert split_groups(heads, 600, 40000, 8, 96) == 3 * 8


def test_pieces_fit_the_list():
    """256 entries in all: the largest count of pieces gives way."""
    assert split_groups([(DENSE, 0, 0)] * 48, 64, 40000, 8, 96) == 48 * 5
    assert split_groups([(DENSE, 0, 0)] * 128, 64, 40000, 8, 96) == 128 * 2
    assert split_groups([(DENSE, 0, 0)] * 32, 64, 40000, 8, 96) == 32 * 8
