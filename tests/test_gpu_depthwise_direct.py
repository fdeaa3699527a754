"""Depthwise 3x3 on 16-bit activations in rows of whole 16-byte vectors on the kernel without LDS (stride 2, small launches of stride 1) against the oracle.

Weights, biases and inputs are fixed-point numbers whose sums of nine are exact in float32: spikes and membranes are the oracle's bit for bit."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import DEV, LIF, dev, gen, spikes, zero_v
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
S = torch.ops.snn_custom
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16


def _layer(C, g):
    return torch.randint(-64, 65, (C, 1, 3, 3), generator=g) / 64.0, torch.randint(-16, 17, (C,), generator=g) / 64.0


def _run(xs, w, b, zero, C, dtype, rs=None, lif=LIF):
    args = (dev(w, dtype), dev(b, dtype), zero, [2, 2], [1, 1], [1, 1], C, *lif, False)
    if rs is not None:
        return S.fused_temporal_conv_add_lif_state_depthwise(xs, [dev(r, dtype) for r in rs], *args)
    return S.fused_temporal_depthwise_conv_lif_state(xs, *args)


# one strip, odd and even heights (the last kernel row inside and outside), strips that end waves and workgroups, several windows of steps
@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("N,C,H,W,T,residual,lif", [(1, 2, 1, 8, 1, False, LIF), (2, 3, 2, 8, 4, True, LIF), (3, 5, 7, 16, 3, False, LIF), (1, 16, 15, 40, 2, True, LIF),
                                                    (2, 24, 64, 64, 4, False, LIF), (1, 8, 56, 56, 20, True, LIF), (1, 7, 9, 24, 4, False, (1.0, -1.0, 3.0))])
def test_rows_of_whole_vectors(hip_ops, dtype, N, C, H, W, T, residual, lif):
    g = gen(31 * H + W)
    xs = [spikes((N, C, H, W), 0.4, g) for _ in range(T)]
    rs = [spikes((N, C, (H + 1) // 2, (W + 1) // 2), 0.3, g) for _ in range(T)] if residual else None
    w, b = _layer(C, g)
    ref = O.temporal_conv_lif(xs, w, b, torch.tensor(0.0), (2, 2), (1, 1), (1, 1), C, *lif, residuals=rs)
    s, v = _run([dev(x, dtype) for x in xs], w, b, zero_v(F32), C, dtype, rs, lif)
    assert torch.equal(s.float().cpu(), ref[0]) and torch.equal(v.cpu(), ref[1])


def test_inputs_that_are_not_aligned_to_vectors(hip_ops):
    """Steps that start four elements into a vector go to the kernel with narrower strips."""
    g = gen(5)
    x = spikes((2, 6, 10, 16), 0.4, g)
    w, b = _layer(6, g)
    ref = O.temporal_conv_lif([x, x], w, b, torch.tensor(0.0), (2, 2), (1, 1), (1, 1), 6, *LIF)
    store = torch.zeros(x.numel() + 8, dtype=BF16, device=DEV)
    shifted = store[4:4 + x.numel()].view(x.shape)
    shifted.copy_(x)
    s, v = _run([shifted, shifted], w, b, zero_v(F32), 6, BF16)
    assert torch.equal(s.float().cpu(), ref[0]) and torch.equal(v.cpu(), ref[1])


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_an_output_sees_its_nine_inputs_only(hip_ops, value):
    """An infinity or NaN in a column or row beside the window does not reach the output."""
    x = torch.zeros((1, 2, 8, 16))
    x[0, 0, 2, 2] = value                        # taps of output rows 1, columns 1 only (even row and column)
    w, b = torch.full((2, 1, 3, 3), 0.25), torch.full((2,), 0.5)
    s, v = _run([dev(x, BF16)], w, b, zero_v(F32), 2, BF16)
    clean = torch.full((1, 2, 4, 8), 0.25)
    got = v.cpu()
    assert torch.equal(torch.where(torch.arange(64).view(1, 2, 4, 8) == 9, clean, got), clean)
    assert s[0, 0, 0, 1, 1].item() == (1.0 if value == float("inf") else 0.0)


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("N,C,H,W,T,residual", [(1, 2, 1, 8, 1, False), (2, 5, 7, 16, 4, True), (1, 16, 15, 40, 3, False), (1, 24, 48, 48, 17, True), (8, 64, 32, 64, 2, False),
                                                (8, 65, 32, 64, 2, False)])
def test_stride_1_without_lds(hip_ops, dtype, N, C, H, W, T, residual):
    """Launches of up to 131072 strips (the last but one) and the first on the tile in LDS: the same dot products in the same order as on row-packed spikes."""
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    g = gen(7 * H + C)
    xs = [spikes((N, C, H, W), 0.4, g) for _ in range(T)]
    rs = [spikes((N, C, H, W), 0.3, g) for _ in range(T)] if residual else None
    w, b = _layer(C, g)
    ref = O.temporal_conv_lif(xs, w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), C, *LIF, residuals=rs)
    dx, dr = [dev(x, dtype) for x in xs], None if rs is None else [dev(r, dtype) for r in rs]
    args = (dev(w, dtype), dev(b, dtype), zero_v(F32), [1, 1], [1, 1], [1, 1], C, *LIF, False)
    s, v = S.fused_temporal_depthwise_conv_lif_state(dx, *args) if rs is None else S.fused_temporal_conv_add_lif_state_depthwise(dx, dr, *args)
    assert torch.equal(s.float().cpu(), ref[0]) and torch.equal(v.cpu(), ref[1])
    noisy = [(x * 0.83).to(dtype) for x in dx]                  # (sums that round)
    args = (dev(w * 0.77, dtype), dev(b, dtype), zero_v(F32), [1, 1], [1, 1], [1, 1], C, *LIF, False)
    s1, v1 = S.fused_temporal_depthwise_conv_lif_state(noisy, *args)
    bits, v2 = B.depthwise_conv_lif_rowbits(noisy, args[0], args[1], LIF)
    assert torch.equal(B.unpack_rowbits(bits, dtype), s1) and torch.equal(v1, v2)


@pytest.mark.parametrize("dtype,vdtype,T,residual,membrane,lif", [
    (BF16, F32, 2, True, True, LIF),
    (F16, F32, 2, True, False, (1.0, 0.25, 2.0)),
    (BF16, BF16, 3, False, True, LIF),               # 16-bit membranes
    (F16, F16, 2, True, True, LIF),
    (BF16, F32, 2, True, True, (1.0, -1.0, 3.0)),    # the general neuron: soft reset, a tau that is no power of two
    (F16, F16, 2, False, False, (1.0, -1.0, 2.0)),
    (F16, F32, 2, False, True, (1.0, 0.0, 1.0)),     # integrate and fire
    (BF16, F32, 18, True, True, LIF),                # two windows of steps
])
def test_stride_1_tile_in_lds(hip_ops, dtype, vdtype, T, residual, membrane, lif):
    """Dense spikes from the tile in LDS, at the fewest strips that it takes (on 256 compute units): residuals, membranes of either dtype, every neuron, several windows."""
    N, C, H, W = 8, 65, 32, 64
    assert N * C * H * W // 8 > 2 * 256 * 256
    g = gen(T + 3 * int(residual))
    xs = [spikes((N, C, H, W), 0.4, g) for _ in range(T)]
    rs = [spikes((N, C, H, W), 0.3, g) for _ in range(T)] if residual else None
    w, b = _layer(C, g)
    v0 = torch.randint(-16, 16, (N, C, H, W), generator=g) / 32.0 if membrane else None
    ref = O.temporal_conv_lif(xs, w, b, torch.tensor(0.0) if v0 is None else v0, (1, 1), (1, 1), (1, 1), C, *lif, residuals=rs)
    vi = zero_v(vdtype) if v0 is None else dev(v0, vdtype)
    args = (dev(w, dtype), dev(b, dtype), vi, [1, 1], [1, 1], [1, 1], C, *lif, False)
    dx = [dev(x, dtype) for x in xs]
    s, v = S.fused_temporal_depthwise_conv_lif_state(dx, *args) if rs is None else S.fused_temporal_conv_add_lif_state_depthwise(dx, [dev(r, dtype) for r in rs], *args)
    assert torch.equal(s.float().cpu(), ref[0]) and torch.equal(v.cpu(), ref[1].to(vdtype))
    assert 0.01 < float(ref[0].mean()) < 0.99
