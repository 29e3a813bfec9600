"""GPU checks of the float32 input route: msa_round_f32 equals torch's own
rounding bit for bit, and an op called with float32 tensors equals the same
call on the explicit roundings, on every route (one launch, torch ops, bf16,
an output that overwrites an input)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _views(dev, D, S):
    g = torch.Generator(dev).manual_seed(D + S)
    x = torch.randn(2, 3, S, D, device=dev, generator=g)
    y = torch.randn(2, S, 5, D, device=dev, generator=g).transpose(1, 2)
    z = torch.randn(2, 3, S, D + 8, device=dev, generator=g)[..., 4:D + 4]
    return x, y, z


@pytest.mark.parametrize("D,S", [(8, 1), (64, 1), (96, 63), (96, 257), (128, 64), (256, 33)])
def test_bits(gpu_device, D, S):
    from minference import _abi

    ts = _views(gpu_device, D, S)
    ts[0].view(-1)[:8] = torch.tensor([0.0, -0.0, 65504.0, -65504.0, 6e-8, 1e-5, float("inf"),
                                       float("nan")])
    assert _abi.round_f32_supported(ts)
    flag = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    outs = _abi.round_f32(ts, flag)
    torch.cuda.synchronize()
    assert int(flag[0]) == 0
    for t, o in zip(ts, outs):
        ref = t.to(torch.float16).contiguous()
        assert o.is_contiguous() and torch.equal(o.view(torch.int16), ref.view(torch.int16))
    ts[1][1, 4, S - 1, D - 1] = -65505.0  # the last element read, just beyond the range
    _abi.round_f32(ts, flag)
    torch.cuda.synchronize()
    assert int(flag[0]) == 1


@pytest.mark.parametrize("big", [False, True])
@pytest.mark.parametrize("D", [96, 92, 80])  # 92: not a multiple of 8, the torch route
def test_op_on_roundings(gpu_device, D, big):
    from minference import streaming_forward

    g = torch.Generator(gpu_device).manual_seed(D)
    q, k, v = (torch.randn(1, 3, 200, D, device=gpu_device, generator=g) for _ in range(3))
    if big:
        v[0, 1, 100, 3] = 1.0e5
    dt = torch.bfloat16 if big else torch.float16
    ref = torch.empty_like(q)
    streaming_forward(q.to(dt), k.to(dt), v.to(dt), 16, 64, out=ref)
    assert torch.equal(streaming_forward(q, k, v, 16, 64), ref)
    got = q.clone()
    assert torch.equal(streaming_forward(got, k, v, 16, 64, out=got), ref)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_fp16_v_needs_no_scale_pass(gpu_device, dtype):
    """The V exponent of an fp16 layer comes from the staging itself: largest
    finite values, Inf and NaN in V, several batches and heads."""
    from minference import dense_attention

    g = torch.Generator(gpu_device).manual_seed(5)
    q, k, v = (torch.randn(2, 3, 130, 64, device=gpu_device, generator=g).to(dtype)
               for _ in range(3))
    v[1, 2, 7, 9] = 65504.0 if dtype == torch.float16 else 1.0e6
    v[0, 1, 3, 5] = float("inf")
    out = dense_attention(q, k, v, causal=False, out=torch.empty(q.shape, device=gpu_device))
    ref = (torch.softmax(q.double() @ k.double().transpose(-1, -2) / 8.0, -1) @ v.double())
    assert torch.isinf(out[0, 1, :, 5]).all()
    fin = torch.isfinite(ref)
    assert torch.equal(fin, torch.isfinite(out))
    scale = v.double().abs().masked_fill(~torch.isfinite(v), 0).amax()
    assert float(((out - ref)[fin]).abs().max()) < 2e-3 * float(scale)


def test_raising_op_waits_for_the_rounding(gpu_device):
    """The launch writes the range flag through its address: an op that raises
    (here: an output of the wrong shape) gives the call back only when the
    launch is done with it."""
    from minference import streaming_forward

    q, k, v = (torch.randn(1, 2, 128, 64, device=gpu_device) for _ in range(3))
    bad = torch.empty(1, 2, 127, 64, device=gpu_device)
    with pytest.raises(ValueError):
        streaming_forward(q, k, v, 16, 64, out=bad)
    torch.cuda.synchronize()
    torch.cuda._sleep(20_000_000)  # the rounding is queued behind some work
    with pytest.raises(ValueError):
        streaming_forward(q, k, v, 16, 64, out=bad)
    assert torch.cuda.current_stream().query()


@pytest.mark.parametrize("big", [False, True])
@pytest.mark.parametrize("S,causal", [(300, True), (32768, True), (32767, True), (23170, False),
                                      (23171, False)])
def test_long_op_runs_once(gpu_device, big, S, causal):
    """From 2^37 operations on the op is queued when its type is known; below,
    it may run a second time on bf16 roundings."""
    from minference.ops.common import accepts_float32

    seen = []

    @accepts_float32(("q", "k", "v"))
    def op(q, k, v, *, causal=True, out=None):
        seen.append(q.dtype)
        assert q.dtype == k.dtype == v.dtype and out.dtype == torch.float32
        return out

    q, k, v = (torch.zeros(1, 1, S, 64, device=gpu_device) for _ in range(3))
    if big:
        k[0, 0, S // 2, 3] = 7.0e4
    op(q, k, v, causal=causal)
    short = 4 * 64 * S * S // (2 if causal else 1) < 2 ** 37
    assert seen == ([torch.float16, torch.bfloat16][0 if not big or short else 1:2 if big else 1])
