"""Convolutions of few output pixels (workgroups of 16 channels x 4, 8 or 16 pixels, columns of timesteps and pixels) against the CPU oracle, and the tiles
of conv_spk_kernel that they replace, which a registered launch choice still selects.

Weights and biases are fixed-point numbers: every sum is exact in float32 in any order, so that spikes are the oracle's and the two kernels agree bit for bit."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import LIF, dev, gen, spikes
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16


@pytest.fixture()
def B(hip_ops):
    from triton_snn_fusion_amd.runtime import hip_blocked_backend
    return hip_blocked_backend


def _operands(T, N, Cin, Cout, H, W, k, s, residual, layout, g):
    x = spikes((T, N, Cin, H, W), 0.3, g)
    if layout == "c8":
        x = x * torch.randint(0, 5, x.shape, generator=g) * 0.25          # averages of spikes
    std = 2.0 ** round(float(torch.log2(torch.tensor(2.5 * (2.0 / (Cin * k * k)) ** 0.5))))
    w = (torch.randn(Cout, Cin, k, k, generator=g) * 16).round().clamp(-64, 64) / 16 * std
    b = (torch.randn(Cout, generator=g) * 2).round() / 16
    p = k // 2
    ho, wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    r = spikes((T, N, Cout, ho, wo), 0.2, g) if residual else None
    return x, w, b, r


CASES = [   # T, N, Cin, Cout, H, W, k, s, dtype, residual, layout, lif, membrane, workgroups expected
    (4, 1, 128, 256, 8, 8, 3, 1, BF16, False, "bits", LIF, False, "1x2x2x16x256"),       # four pixels, five fragments a wave
    (4, 2, 256, 256, 7, 7, 3, 1, F16, True, "bits", LIF, True, "1x7x1x16x224"),          # eight, seven of them used; nine fragments
    (4, 1, 512, 512, 4, 4, 3, 1, BF16, True, "bits", LIF, False, "1x2x2x16x128"),        # 18 fragments
    (4, 4, 256, 256, 8, 8, 3, 1, BF16, True, "bits", LIF, False, "1x4x4x16x256"),        # sixteen pixels
    (4, 5, 512, 500, 2, 2, 3, 1, BF16, True, "c8", (1.0, -1.0, 3.0), True, "1x2x2x16x160"),   # planes of four pixels, soft reset, a last tile of four channels
    (4, 9, 512, 512, 1, 2, 1, 1, F16, False, "bits", LIF, True, "2x1x2x16x160"),         # whole planes of several images, the last workgroup half empty
    (3, 1, 72, 40, 9, 7, 3, 1, BF16, True, "bits", LIF, True, None),                     # three steps, an odd number of channel groups
    (2, 1, 256, 128, 6, 5, 3, 1, F16, True, "bits", LIF, True, None),                    # two steps
    (9, 1, 128, 136, 6, 6, 3, 2, BF16, True, "bits", (1.0, 0.25, 4.0), True, None),      # three windows, the last of one step; stride 2
    (8, 1, 64, 128, 8, 8, 5, 1, BF16, False, "c8", LIF, False, None),                    # 25 taps: an odd number of entries per wave
    (4, 1, 1024, 64, 5, 3, 3, 1, BF16, False, "bits", LIF, False, None),                 # more fragments than fly at once
]


@pytest.mark.parametrize("T,N,Cin,Cout,H,W,k,s,dtype,residual,layout,lif,membrane,workgroups", CASES)
def test_few_pixels(B, T, N, Cin, Cout, H, W, k, s, dtype, residual, layout, lif, membrane, workgroups):
    g = gen(Cin + Cout + 7 * H + T)
    x, w, b, r = _operands(T, N, Cin, Cout, H, W, k, s, residual, layout, g)
    p = k // 2
    v0 = torch.randint(-16, 16, (N, Cout, (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1), generator=g) / 32.0 if membrane else None
    ref = O.temporal_conv_lif([x[t] for t in range(T)], w, b, torch.tensor(0.0) if v0 is None else v0, (s, s), (p, p), (1, 1), 1, *lif,
                              residuals=None if r is None else [r[t] for t in range(T)])
    xb = B.from_dense(dev(x, dtype), B.BITS if layout == "bits" else B.C8)
    rb = None if r is None else B.from_dense(dev(r, dtype), B.BITS)

    def call():
        out, v = B.conv_lif_blocked(xb, dev(w, dtype), dev(b, dtype), [s, s], [p, p], lif, residual=rb, v_init=None if v0 is None else dev(v0, torch.float32), want_v=True)
        return B.to_dense(out).float().cpu(), v.cpu(), B.last_conv_plan()

    sp, v, plan = call()
    assert "few" in plan and workgroups in (None, plan["few"]), plan
    near = (ref[2] - lif[0]).abs() < 1e-5                                  # (a tau of 3 and rounded membranes: neurons at the threshold)
    assert not ((sp != ref[0]) & ~near).any()
    assert 0.01 < float(ref[0].mean()) < 0.9
    same = (sp == ref[0]).all(0)
    assert torch.allclose(v[same], ref[1][same], rtol=1e-5, atol=1e-5)
    # The tiles of conv_spk_kernel, by a registered patch: the same spikes and membranes.
    key = (T, N, Cin, H, W, Cout, k, k, s, s, p, p, 0)
    B.register_tuned_plan(key, int(plan["tile"].split("x")[2]), 0, 0)
    try:
        sp2, v2, plan2 = call()
    finally:
        B.register_tuned_plan(key, 0, 0, 0)
    assert "few" not in plan2, plan2
    assert torch.equal(sp, sp2) and torch.allclose(v, v2, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("Cin,Cout,H,W,N,dtype", [(256, 256, 8, 8, 1, BF16), (128, 64, 6, 10, 2, F16), (512, 512, 4, 4, 3, BF16), (512, 512, 2, 2, 2, BF16)])
def test_average_pool_of_few_pixels(B, Cin, Cout, H, W, N, dtype):
    g = gen(Cin + H)
    x, w, b, _ = _operands(4, N, Cin, Cout, H, W, 3, 1, False, "bits", g)
    ref = O.temporal_conv_lif([x[t] for t in range(4)], w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), 1, *LIF)
    pooled, v = B.conv_lif_blocked_avgpool(B.from_dense(dev(x, dtype), B.BITS), dev(w, dtype), dev(b, dtype), [1, 1], [1, 1], LIF, want_v=True)
    assert "few" in B.last_conv_plan(), B.last_conv_plan()
    want = torch.nn.functional.avg_pool2d(ref[0].flatten(0, 1), 2)
    assert torch.equal(B.to_dense(pooled).float().cpu().flatten(0, 1), want) and torch.equal(v.cpu(), ref[1])


@pytest.mark.parametrize("dtype,vdtype", [(BF16, BF16), (F16, torch.float32), (F16, F16)])
def test_dense_tensors_of_few_pixels(hip_ops, dtype, vdtype):
    """The dense route: membranes of either dtype, through several windows, rounded once at the end."""
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    S = torch.ops.snn_custom
    g = gen(91)
    T, N, Cin, Cout, H, W = 6, 2, 256, 136, 5, 7
    x, w, b, r = _operands(T, N, Cin, Cout, H, W, 3, 1, True, "bits", g)
    v0 = torch.randint(-16, 16, (N, Cout, H, W), generator=g) / 32.0
    ref = O.temporal_conv_lif([x[t] for t in range(T)], w, b, v0, (1, 1), (1, 1), (1, 1), 1, *LIF, residuals=[r[t] for t in range(T)])
    s, v = S.fused_temporal_conv_add_lif_state([dev(x[t], dtype) for t in range(T)], [dev(r[t], dtype) for t in range(T)], dev(w, dtype), dev(b, dtype),
                                               dev(v0, vdtype), [1, 1], [1, 1], [1, 1], 1, *LIF, False)
    assert "few" in CB.last_conv_plan(), CB.last_conv_plan()
    assert torch.equal(s.float().cpu(), ref[0]) and torch.equal(v.cpu(), ref[1].to(vdtype))


@pytest.mark.parametrize("lif", [(1.0, -1.0, 2.0), LIF, (1.0, 0.25, 2.0)])
@pytest.mark.parametrize("T", [4, 5])
def test_rounding_of_the_charge(B, lif, T):
    """Membranes of 24 bits, on which (v + x) / 2 and v + (x - v) / 2 round differently: the charge of the tiles of conv_spk_kernel for either reset, with a soft
    reset the oracle's own."""
    g = gen(17)
    Cin, Cout, H = 128, 64, 6
    x, w, b, _ = _operands(T, 1, Cin, Cout, H, H, 3, 1, False, "bits", g)
    v0 = torch.randn((1, Cout, H, H), generator=g) * 0.7
    ref = O.temporal_conv_lif([x[t] for t in range(T)], w, b, v0, (1, 1), (1, 1), (1, 1), 1, *lif)
    first = torch.nn.functional.conv2d(x[0], w, b, padding=1)
    differ = float(((v0 + first) * 0.5 != v0 + (first - v0) * 0.5).float().mean())
    assert differ > 0.02, differ                                           # the two forms are told apart
    xb = B.from_dense(dev(x, BF16), B.BITS)

    def call():
        out, v = B.conv_lif_blocked(xb, dev(w, BF16), dev(b, BF16), [1, 1], [1, 1], lif, v_init=dev(v0, torch.float32), want_v=True)
        return B.to_dense(out).float().cpu(), v.cpu(), B.last_conv_plan()

    sp, v, plan = call()
    assert "few" in plan, plan
    key = (T, 1, Cin, H, H, Cout, 3, 3, 1, 1, 1, 1, 0)
    B.register_tuned_plan(key, int(plan["tile"].split("x")[2]), 0, 0)
    try:
        sp2, v2, plan2 = call()
    finally:
        B.register_tuned_plan(key, 0, 0, 0)
    assert "few" not in plan2, plan2
    assert torch.equal(sp, sp2) and torch.equal(v, v2)
    if lif[1] < 0:
        assert torch.equal(sp, ref[0]) and torch.equal(v, ref[1])


@pytest.mark.parametrize("Cin,k,value", [(72, 3, float("inf")), (72, 3, float("nan")), (200, 1, float("inf")), (200, 1, float("nan")), (64, 5, float("inf"))])
def test_an_output_sees_its_own_inputs_only(B, Cin, k, value):
    """An infinity or NaN reaches the outputs whose window holds it and no other: neither through the entry that an odd number leaves without a partner, nor through
    padding, an odd number of channel groups or pixels beyond the plane."""
    g = gen(Cin + k)
    T, Cout, H, W = 4, 48, 5, 7
    x, w, b, _ = _operands(T, 1, Cin, Cout, H, W, k, 1, False, "c8", g)
    w = torch.where(w == 0, torch.full_like(w, w.abs().max().item()), w).abs()       # (no product is 0 x infinity, all have one sign)
    xb = B.from_dense(dev(x, BF16), B.C8)
    args = (dev(w, BF16), dev(b, BF16), [1, 1], [k // 2, k // 2], LIF)
    sp, v = B.conv_lif_blocked(xb, *args, want_v=True)
    assert "few" in B.last_conv_plan(), B.last_conv_plan()
    bad = x.clone()
    bad[1, 0, Cin - 1, 4, 6] = value                                                 # the last channel of the last pixel
    sp2, v2 = B.conv_lif_blocked(B.from_dense(dev(bad, BF16), B.C8), *args, want_v=True)
    seen = torch.zeros((H, W), dtype=torch.bool)
    seen[max(0, 4 - k // 2):, max(0, 6 - k // 2):] = True
    one, two = B.to_dense(sp).float().cpu(), B.to_dense(sp2).float().cpu()
    assert torch.equal(v.cpu()[:, :, ~seen], v2.cpu()[:, :, ~seen]) and torch.equal(one[..., ~seen], two[..., ~seen]) and torch.equal(one[0], two[0])
    fired = two[1, 0][:, seen]
    assert bool((fired == (1.0 if value == float("inf") else 0.0)).all()), fired
