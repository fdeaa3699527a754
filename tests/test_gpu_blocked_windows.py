"""Blocked convolutions of more timesteps than a window holds, bit-packed in and out: the straight-line epilogue passes the membrane from
window to window. Against the CPU oracle for every way the waves of a workgroup share a tile, with windows of four timesteps (the last one of one to
four) and of three (five, six and nine timesteps)."""
import pytest
import torch

from helpers import LIF, check, dev, gen, q, spikes
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("Cin,Cout,H,W,N,T,window,dtype,residual,layout,waves,tile", [
    (64, 64, 56, 56, 9, 5, 3, BF16, True, "bits", "8x1x2", 64),       # two waves per tile; windows of three, the last one of two steps
    (64, 64, 56, 56, 9, 13, 4, BF16, True, "bits", "8x1x2", 64),      # windows of four, the last one of one step
    (16, 64, 40, 40, 46, 6, 3, BF16, True, "bits", "8x1x1", 64),      # a wave per tile, several rounds
    (16, 64, 40, 40, 46, 10, 4, BF16, True, "bits", "8x1x1", 64),     # windows of four, the last one of two steps
    (16, 72, 40, 40, 20, 8, 4, F16, False, "c8", "8x1x1", 64),        # blocked inputs; eight channels in the last tile
    (256, 128, 14, 14, 24, 7, 4, BF16, True, "bits", "8x1x4", 64),    # four waves per tile; a last window of three steps
    (256, 128, 14, 14, 24, 13, 4, BF16, True, "bits", "8x1x4", 64),
    (512, 512, 7, 7, 9, 6, 3, BF16, False, "bits", "8x1x8", 64),      # eight
    (512, 512, 7, 7, 9, 10, 4, BF16, False, "bits", "8x1x8", 64),
    (128, 40, 8, 8, 1, 16, 4, BF16, True, "bits", "8x1x8", 32),       # tiles of 32 channels, four windows
    (128, 40, 8, 8, 1, 13, 4, BF16, True, "bits", "8x1x8", 32),
    (64, 96, 9, 11, 2, 9, 3, F16, True, "c8", "8x1x4", 32),
    (64, 96, 9, 11, 2, 10, 4, F16, True, "c8", "8x1x4", 32),
])
def test_membrane_passes_from_window_to_window(snnf_lib, Cin, Cout, H, W, N, T, window, dtype, residual, layout, waves, tile):
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    g = gen(7000 + Cin + T)
    x = torch.stack([spikes((N, Cin, H, W), 0.25, g) for _ in range(T)])
    w, b = q(torch.randn(Cout, Cin, 3, 3, generator=g) * 2.0 * (2.0 / (Cin * 9)) ** 0.5, dtype), q(torch.randn(Cout, generator=g) * 0.1, dtype)
    rs = torch.stack([spikes((N, Cout, H, W), 0.25, g) for _ in range(T)]) if residual else None
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), 1, *LIF, residuals=list(rs) if residual else None)
    out, v = B.conv_lif_blocked(B.from_dense(dev(x, dtype), B.BITS if layout == "bits" else B.C8), dev(w, dtype), dev(b, dtype), [1, 1], [1, 1], LIF,
                                residual=B.from_dense(dev(rs, dtype), B.BITS) if residual else None, out_layout=B.BITS, want_v=True)
    plan = B.last_conv_plan()
    assert int(plan["variant"]) >= 60 and int(plan["window"]) == window, plan
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert (plan["waves"], int(plan["oc_tile"])) == (waves, tile), plan
    check(B.to_dense(out), v, ref, what=f"{Cin}->{Cout} {H}x{W} T={T}")


@pytest.mark.parametrize("Cin,Cout,H,W,N,window", [
    (16, 96, 40, 40, 46, 4),      # a wave per tile: windows of four, four and one
    (24, 120, 58, 58, 13, 4),
    (48, 96, 14, 14, 4, 3),       # waves that share a tile: three of three
])
def test_nine_steps_of_1x1(snnf_lib, Cin, Cout, H, W, N, window):
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    g = gen(7100 + Cin)
    x = torch.stack([spikes((N, Cin, H, W), 0.25, g) for _ in range(9)])
    w, b = q(torch.randn(Cout, Cin, 1, 1, generator=g) * 2.0 * (2.0 / Cin) ** 0.5, BF16), q(torch.randn(Cout, generator=g) * 0.1, BF16)
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (0, 0), (1, 1), 1, *LIF)
    out, v = B.conv_lif_blocked(B.from_dense(dev(x, BF16), B.BITS), dev(w, BF16), dev(b, BF16), [1, 1], [0, 0], LIF, out_layout=B.BITS, want_v=True)
    plan = B.last_conv_plan()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert int(plan["window"]) == window, plan
    check(B.to_dense(out), v, ref, what=f"{Cin}->{Cout} {H}x{W} T=9")


SOFT = (1.0, -1.0, 2.0)


@pytest.mark.parametrize("Cin,Cout,H,W,k,N,T,dtype,residual,layout,lif", [
    (64, 8, 28, 28, 3, 73, 6, BF16, True, "bits", LIF),       # one group of channels, several rounds and windows
    (16, 32, 40, 40, 3, 5, 4, F16, True, "c8", LIF),
    (16, 24, 9, 11, 5, 3, 1, BF16, True, "bits", LIF),        # one step
    (16, 96, 8, 8, 3, 3, 2, BF16, False, "bits", LIF),        # three tiles of 32 channels, two steps
    (16, 72, 14, 14, 1, 2, 4, F16, True, "bits", LIF),        # the last of them with 8
    (16, 20, 13, 7, 3, 2, 7, BF16, True, "c8", SOFT),         # the general epilogue, half a group of channels
])
def test_narrow_tiles_of_one_wave(snnf_lib, Cin, Cout, H, W, k, N, T, dtype, residual, layout, lif):
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    g = gen(7300 + Cin + Cout + T)
    x = torch.stack([spikes((N, Cin, H, W), 0.25, g) for _ in range(T)])
    w, b = q(torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5, dtype), q(torch.randn(Cout, generator=g) * 0.1, dtype)
    rs = torch.stack([spikes((N, Cout, H, W), 0.25, g) for _ in range(T)]) if residual else None
    p = k // 2
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (p, p), (1, 1), 1, *lif, residuals=list(rs) if residual else None)
    out, v = B.conv_lif_blocked(B.from_dense(dev(x, dtype), B.BITS if layout == "bits" else B.C8), dev(w, dtype), dev(b, dtype), [1, 1], [p, p], lif,
                                residual=B.from_dense(dev(rs, dtype), B.BITS) if residual else None, out_layout=B.BITS, want_v=True)
    plan = B.last_conv_plan()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert (plan["waves"], int(plan["oc_tile"])) == ("8x1x1", 32), plan
    check(B.to_dense(out), v, ref, what=f"{Cin}->{Cout} {H}x{W} T={T}")


@pytest.mark.parametrize("Cin,Cout,H,k,s,N,T,out,lif", [
    (3, 64, 32, 3, 1, 2, 4, "bits", LIF),
    (3, 96, 20, 7, 2, 1, 6, "bits", LIF),                     # three tiles of 32 channels, steps in a loop
    (1, 8, 9, 3, 1, 3, 2, "c8", LIF),                         # the general epilogue
    (3, 64, 32, 3, 1, 70, 8, "bits", LIF),                    # 2240 patches: tiles of 64 channels again
    (2, 64, 16, 3, 1, 3, 4, "pooled", LIF),
])
def test_narrow_tiles_of_a_frame(snnf_lib, Cin, Cout, H, k, s, N, T, out, lif):
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    g = gen(7350 + Cout + T)
    frame = q(torch.randn(N, Cin, H, H, generator=g), BF16)
    w, b = q(torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5, BF16), q(torch.randn(Cout, generator=g) * 0.1, BF16)
    p = k // 2
    ref = O.temporal_conv_lif([frame] * T, w, b, torch.tensor(0.0), (s, s), (p, p), (1, 1), 1, *lif)
    x = B.input_frame(dev(frame, BF16), T)
    if out == "pooled":
        got = B.to_dense(B.conv_lif_blocked_avgpool(x, dev(w, BF16), dev(b, BF16), [s, s], [p, p], lif)[0]).float().cpu()
        want = torch.stack([torch.nn.functional.avg_pool2d(t, 2) for t in ref[0]])
        assert float((got != want).float().mean()) <= 1e-3
    else:
        o, v = B.conv_lif_blocked(x, dev(w, BF16), dev(b, BF16), [s, s], [p, p], lif, out_layout=B.BITS if out == "bits" else B.C8, want_v=True)
        check(B.to_dense(o), v, ref, what=f"{Cin}->{Cout} {H}x{H} T={T}")
    plan = B.last_conv_plan()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert int(plan["oc_tile"]) == (64 if N == 70 else 32), plan
