"""One dense frame of at most eight channels for all timesteps, dense spikes out, on the blocked kernel, against the oracle and against equal frames per timestep.

Weights, biases and pixels are fixed-point numbers: sums are exact in float32 in any order, spikes and membranes are the oracle's bit for bit."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import DEV, LIF, dev, gen
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,N,T,dtype,vdtype,membrane", [
    (3, 64, 64, 64, 7, 2, 2, 4, BF16, F32, False),       # patches of one row of 32
    (3, 64, 32, 32, 3, 1, 1, 2, F16, F32, True),
    (3, 64, 48, 224, 7, 2, 1, 16, BF16, F32, False),     # two rows of 16, as many steps as a launch takes
    (1, 6, 9, 31, 3, 1, 2, 3, BF16, F32, True),          # six channels, a patch that hangs over the plane
    (8, 37, 7, 5, 5, 1, 3, 5, F16, F32, True),           # an odd number of channels, planes of less than a patch
    (4, 96, 50, 50, 3, 2, 2, 4, BF16, BF16, True),       # a 16-bit membrane
    (2, 72, 13, 17, 1, 1, 2, 6, F16, F32, False),        # 1x1
])
def test_dense_frame(hip_ops, Cin, Cout, H, W, k, s, N, T, dtype, vdtype, membrane):
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    S = torch.ops.snn_custom
    g = gen(Cin + 10 * Cout + H)
    p = k // 2
    x = torch.randint(-32, 33, (N, Cin, H, W), generator=g) / 16.0
    w = torch.randint(-16, 17, (Cout, Cin, k, k), generator=g) / 16.0 / k
    w = (w * 32).round() / 32
    b = torch.randint(-8, 9, (Cout,), generator=g) / 16.0
    v0 = torch.randint(-16, 16, (N, Cout, (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1), generator=g) / 32.0 if membrane else None
    ref = O.temporal_conv_lif([x] * T, w, b, torch.tensor(0.0) if v0 is None else v0, (s, s), (p, p), (1, 1), 1, *LIF)
    dx, vi = dev(x, dtype), torch.zeros((), device=DEV, dtype=vdtype) if v0 is None else dev(v0, vdtype)
    args = (dev(w, dtype), dev(b, dtype), vi, [s, s], [p, p], [1, 1], 1, *LIF, False)
    sp, v = S.fused_temporal_conv_lif_state([dx] * T, *args)
    plan = CB.last_conv_plan()
    assert plan["route"] == "frame" and plan["ran"] == "blocked" and int(plan["window"]) == T, plan
    assert torch.equal(sp.float().cpu(), ref[0]) and 0.01 < float(ref[0].mean()) < 0.9
    # (a neuron that keeps charging ends with more bits than float32 has: charged as v + (x - v) / 2, as by the oracle)
    assert torch.equal(v.cpu(), ref[1].to(vdtype))
    sp2, v2 = S.fused_temporal_conv_lif_state([dx.clone() for _ in range(T)], *args)
    assert torch.equal(sp, sp2) and torch.allclose(v.float(), v2.float(), rtol=1e-6 if vdtype == F32 else 2.0 ** -7, atol=1e-6)


@pytest.mark.parametrize("lif,residual,dtype,Cin", [((1.0, -1.0, 2.0), False, BF16, 3), ((1.0, 0.0, 3.0), False, BF16, 3), (LIF, True, BF16, 3), (LIF, False, F32, 3), (LIF, False, BF16, 16)])
def test_frames_that_stay_on_the_dense_kernels(hip_ops, lif, residual, dtype, Cin):
    """Other neurons, residuals, float32 and more than eight channels."""
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    S = torch.ops.snn_custom
    g = gen(Cin)
    x, w, b = torch.randn((2, Cin, 16, 16), generator=g), torch.randn((64, Cin, 3, 3), generator=g) * 0.3, torch.zeros(64)
    args = (dev(w, dtype), dev(b, dtype), torch.zeros((), device=DEV), [1, 1], [1, 1], [1, 1], 1, *lif, False)
    dx = dev(x, dtype)
    if residual:
        S.fused_temporal_conv_add_lif_state([dx] * 4, [torch.zeros((2, 64, 16, 16), device=DEV, dtype=dtype)] * 4, *args)
    else:
        S.fused_temporal_conv_lif_state([dx] * 4, *args)
    assert CB.last_conv_plan().get("route") != "frame", CB.last_conv_plan()


@pytest.mark.parametrize("T,N,Cin,Cout,H,W,k,s,frame", [
    (4, 19, 3, 64, 224, 224, 7, 2, True),      # a stem of 61 million outputs
    (4, 20, 3, 64, 224, 224, 7, 2, False),     # of 64
    (8, 45, 4, 96, 96, 25, 1, 1, True),        # 1x1 on the time-outer kernel, 83 million
    (8, 50, 4, 96, 96, 25, 1, 1, False),       # 92
    (4, 30, 3, 64, 112, 112, 3, 1, True),      # whole tiles of stride 1, 96 million
])
def test_line_of_large_outputs(hip_ops, T, N, Cin, Cout, H, W, k, s, frame):
    """Large first layers stay on the dense kernel where that is the faster one; either way an image has the spikes that it has alone."""
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    S = torch.ops.snn_custom
    x = torch.randint(-32, 33, (N, Cin, H, W), device=DEV, dtype=torch.int8).to(BF16) / 16
    w = (torch.randint(-16, 17, (Cout, Cin, k, k), device=DEV, dtype=torch.int8).to(BF16) / 64)
    b = torch.zeros(Cout, device=DEV, dtype=BF16)
    args = (w, b, torch.zeros((), device=DEV), [s, s], [k // 2, k // 2], [1, 1], 1, *LIF, False)
    sp, _ = S.fused_temporal_conv_lif_state([x] * T, *args)
    assert (CB.last_conv_plan().get("route") == "frame") == frame, CB.last_conv_plan()
    alone, _ = S.fused_temporal_conv_lif_state([x[-1:]] * T, *args)          # (one image: always the blocked kernel)
    assert CB.last_conv_plan().get("route") == "frame"
    assert torch.equal(sp[:, -1:], alone) and 0.0 < float(alone.float().mean()) < 1.0


@pytest.mark.parametrize("Cin,Cout,H,k,s,N,T,dtype,same_bits", [
    (3, 64, 32, 3, 1, 2, 4, BF16, True),       # whole tiles of the matrix kernel, the same order of products
    (3, 64, 32, 3, 1, 2, 8, F16, True),
    (3, 64, 224, 7, 2, 2, 4, BF16, False),     # (a small batch of strided layers takes the copy route per timestep)
    (8, 64, 56, 3, 1, 4, 4, F16, False),       # whole tiles, another order
    (3, 64, 33, 3, 1, 2, 4, BF16, False),      # planes that tiles do not divide: the copy route per timestep
])
def test_equal_frames_with_sums_that_round(hip_ops, Cin, Cout, H, k, s, N, T, dtype, same_bits):
    """One frame T times against T equal frames on operands whose sums round: the same bits where both add in the same order, else within what the order of additions
    can change - n products of magnitude sum A differ by up to 2 n 2^-24 A between two orders, and a neuron's halvings sum such differences to less than one of them."""
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    S = torch.ops.snn_custom
    g = gen(7 * Cin + H)
    x = dev(torch.randn((N, Cin, H, H), generator=g), dtype)
    w = dev(torch.randn((Cout, Cin, k, k), generator=g) * 3 * (2 / (Cin * k * k)) ** 0.5, dtype)
    b = dev(torch.randn(Cout, generator=g) * 0.1, dtype)
    args = (w, b, torch.zeros((), device=DEV), [s, s], [k // 2, k // 2], [1, 1], 1, *LIF, False)
    sp, v = S.fused_temporal_conv_lif_state([x] * T, *args)
    assert CB.last_conv_plan().get("route") == "frame", CB.last_conv_plan()
    sp2, v2 = S.fused_temporal_conv_lif_state([x.clone() for _ in range(T)], *args)
    assert CB.last_conv_plan().get("route") != "frame", CB.last_conv_plan()
    if same_bits:
        assert "route" not in CB.last_conv_plan(), CB.last_conv_plan()
        assert torch.equal(sp, sp2) and torch.equal(v, v2)
    total = torch.nn.functional.conv2d(x.float().cpu().abs(), w.float().cpu().abs(), b.float().cpu().abs(), s, k // 2)
    bound = (2 * (Cin * k * k + 1) + 4 * T) * 2.0 ** -24 * (total + 1.0)     # (four roundings of a charge per step, of values up to A + 1)
    same = (sp == sp2).all(0).cpu()
    assert float((~same).float().mean()) < 1e-4                              # neurons at the threshold
    assert bool(((v - v2).cpu().abs() <= bound)[same].all())
