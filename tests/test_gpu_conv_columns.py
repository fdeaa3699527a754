"""1x1 convolutions without a neuron on their own kernel: strides, ragged tiles of pixels and channels, odd numbers of channel groups, against float64."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import DEV, dev, gen, q

pytestmark = pytest.mark.gpu

BF16, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("Cin,Cout,H,W,s,T,N", [
    (8, 1, 1, 1, 1, 1, 1),             # a single output
    (8, 24, 5, 7, 1, 2, 3),            # one group: half of its pair is not there; K is not shared; one fragment of channels
    (24, 33, 6, 5, 2, 3, 2),           # two fragments, one channel in the second
    (56, 64, 9, 9, 2, 4, 1),           # seven groups on four waves
    (64, 128, 8, 8, 1, 1, 4),          # whole tiles
    (72, 100, 7, 9, 3, 5, 2),          # stride 3, the last wave has less of K; four fragments, four channels in the last
    (136, 129, 10, 4, 2, 2, 5),        # a second tile of channels of one channel
    (512, 200, 4, 4, 2, 16, 9),        # a long K
    (1024, 40, 3, 3, 1, 2, 2),
    (32, 520, 2, 33, 2, 4, 1),         # five tiles of channels; a step's columns end inside a tile
])
@pytest.mark.parametrize("dtype", [BF16, F16])
def test_against_float64(hip_ops, Cin, Cout, H, W, s, T, N, dtype):
    """One rounding of the result (half a unit in the last place) on top of the float32 sums' own error, at most Cin + 1 roundings of the sum of magnitudes."""
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(Cin + Cout + H)
    x = [q(torch.randn(N, Cin, H, W, generator=g), dtype) for _ in range(T)]
    w, b = q(torch.randn(Cout, Cin, 1, 1, generator=g) / Cin ** 0.5, dtype), q(torch.randn(Cout, generator=g), dtype)
    steps = [dev(t, dtype) for t in reversed(x)][::-1]                     # descending in memory, not one tensor
    out = CB.run_hip_temporal_conv_bias(steps, dev(w, dtype), dev(b, dtype), [s, s], [0, 0])
    plan = CB.last_conv_plan()
    assert (plan["kernel"], plan.get("ran")) == ("matrix", "blocked" if plan.get("route") == "c8" else "columns"), plan
    assert plan.get("route") != "c8" or Cin >= 432, plan                   # (a long K on masked tiles has the blocked route)
    conv = torch.nn.functional.conv2d
    ref = torch.stack([conv(t.double(), w.double(), b.double(), s) for t in x])
    size = torch.stack([conv(t.double().abs(), w.double().abs(), b.double().abs(), s) for t in x])
    bound = ref.abs() * 2.0 ** (-8 if dtype == BF16 else -11) + (Cin + 1) * 2.0 ** -24 * size + 2.0 ** -24
    assert bool(((out.double().cpu() - ref).abs() <= bound).all())


@pytest.mark.parametrize("Cin,Cout,H,s,N,columns", [(64, 128, 56, 2, 16, True), (256, 512, 14, 2, 80, True), (256, 512, 14, 2, 120, False), (64, 128, 56, 1, 4, True), (64, 128, 56, 1, 8, False)])
def test_line(hip_ops, Cin, Cout, H, s, N, columns):
    """Layers of many outputs stay on the matrix kernel; either way an image has the sums that it has alone."""
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    x = (torch.rand(4, N, Cin, H, H, device=DEV) < 0.2).to(BF16)
    w, b = torch.randint(-8, 9, (Cout, Cin, 1, 1), device=DEV).to(BF16) / 16, torch.zeros(Cout, device=DEV, dtype=BF16)
    out = CB.run_hip_conv_bias_frames(x, w, b, [s, s], [0, 0])
    assert (CB.last_conv_plan().get("ran") == "columns") == columns, CB.last_conv_plan()
    assert torch.equal(out[:, -1:], CB.run_hip_conv_bias_frames(x[:, -1:].contiguous(), w, b, [s, s], [0, 0]))
