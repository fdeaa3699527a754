"""Blocked convolutions of timesteps that windows of three or one window of five or six hold: bit-packed layers and dense calls against the CPU oracle,
where the waves of a workgroup share a tile and where they don't, with a last window of two or three steps."""
import pytest
import torch

from helpers import DEV, LIF, check, dev, gen, q, spikes
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
SOFT = (1.0, -1.0, 2.0)


def _layer(Cin, Cout, H, W, k, N, T, dtype, residual, seed):
    g = gen(seed)
    x = torch.stack([spikes((N, Cin, H, W), 0.25, g) for _ in range(T)])
    w, b = q(torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5, dtype), q(torch.randn(Cout, generator=g) * 0.1, dtype)
    rs = torch.stack([spikes((N, Cout, H, W), 0.25, g) for _ in range(T)]) if residual else None
    return x, w, b, rs


@pytest.mark.parametrize("Cin,Cout,H,W,k,N,T,dtype,residual,layout,want_v,lif,steps", [
    (64, 64, 56, 56, 3, 9, 3, BF16, True, "bits", False, LIF, 3),     # one window of three, the usual tile: two waves share it
    (64, 64, 56, 56, 3, 14, 3, BF16, True, "bits", True, LIF, 3),     # a wave per tile, with a membrane
    (16, 72, 40, 40, 3, 30, 3, F16, False, "c8", False, LIF, 3),      # several rounds, eight channels in the last tile
    (64, 64, 20, 20, 3, 60, 5, BF16, True, "bits", True, LIF, 3),     # a last window of two steps
    (128, 64, 14, 14, 3, 40, 6, F16, False, "c8", True, LIF, 3),
    (16, 20, 40, 40, 5, 30, 9, BF16, True, "bits", True, SOFT, 3),    # three windows, the general epilogue, half a group of channels
    (64, 96, 24, 24, 3, 4, 5, BF16, True, "bits", True, LIF, 6),      # one window: four waves a tile, a step beyond T
    (64, 40, 24, 23, 3, 6, 6, F16, False, "c8", True, LIF, 6),        # eight channels in the last tile
    (32, 160, 28, 20, 3, 9, 6, BF16, False, "bits", True, LIF, 6),    # two waves a tile: each finishes two quads
    (176, 64, 16, 16, 3, 8, 6, BF16, True, "bits", True, LIF, 6),     # eight
    (32, 44, 24, 24, 3, 8, 5, BF16, True, "bits", True, SOFT, 6),     # the general epilogue
])
def test_internal_layouts(snnf_lib, Cin, Cout, H, W, k, N, T, dtype, residual, layout, want_v, lif, steps):
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    x, w, b, rs = _layer(Cin, Cout, H, W, k, N, T, dtype, residual, 9000 + Cin + Cout + T)
    p = k // 2
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (p, p), (1, 1), 1, *lif, residuals=list(rs) if residual else None)
    out, v = B.conv_lif_blocked(B.from_dense(dev(x, dtype), B.BITS if layout == "bits" else B.C8), dev(w, dtype), dev(b, dtype), [1, 1], [p, p], lif,
                                residual=B.from_dense(dev(rs, dtype), B.BITS) if residual else None, out_layout=B.BITS, want_v=want_v)
    plan = B.last_conv_plan()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert int(plan["variant"]) % 10 == steps, plan
    check(B.to_dense(out), v if want_v else ref[1], ref, what=f"{Cin}->{Cout} {H}x{W} T={T}")


@pytest.mark.parametrize("Cin,Cout,H,W,k,N,T,dtype,residual,v_dtype,start,steps", [
    (72, 104, 27, 35, 3, 5, 6, F16, True, F16, False, 3),             # windows of three with a 16-bit membrane
    (24, 30, 13, 17, 3, 40, 3, BF16, True, F32, True, 3),             # single channels masked
    (64, 64, 24, 24, 3, 4, 6, BF16, True, BF16, True, 6),             # one window from and to a 16-bit membrane
    (20, 33, 15, 17, 3, 12, 5, F16, True, F32, True, 6),
    (48, 56, 13, 13, 5, 4, 5, F32, True, F32, False, 3),              # fp32 tensors
    (32, 40, 14, 14, 3, 6, 3, F32, False, F32, True, 3),
])
def test_dense_tensors(hip_ops, snnf_lib, Cin, Cout, H, W, k, N, T, dtype, residual, v_dtype, start, steps):
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    x, w, b, rs = _layer(Cin, Cout, H, W, k, N, T, dtype, residual, 9100 + Cin + Cout + T)
    p = k // 2
    v0 = q(torch.randn(N, Cout, H, W, generator=gen(9)) * 0.3, v_dtype) if start else None
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0) if v0 is None else v0, (1, 1), (p, p), (1, 1), 1, *LIF, residuals=list(rs) if residual else None)
    zero = torch.zeros((), dtype=F32, device=DEV) if v_dtype == F32 else torch.zeros(())
    args = (dev(w, dtype), dev(b, dtype), zero if v0 is None else dev(v0, v_dtype), [1, 1], [p, p], [1, 1], 1, *LIF, False)
    xs = [dev(t, dtype) for t in x]
    S = torch.ops.snn_custom
    sp, v = S.fused_temporal_conv_add_lif_state(xs, [dev(t, dtype) for t in rs], *args) if residual else S.fused_temporal_conv_lif_state(xs, *args)
    plan = CB.last_conv_plan()
    assert v.dtype == v_dtype and plan.get("ran") == "blocked", plan
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert int(plan["variant"]) % 10 == steps, plan
    check(sp, v, ref, v_dtype=v_dtype, what=f"{Cin}->{Cout} {H}x{W} T={T}")


@pytest.mark.parametrize("Cin,Cout,H,N,T", [(32, 64, 14, 8, 3), (64, 128, 28, 40, 6), (32, 48, 7, 3, 5)])
def test_shortcut(snnf_lib, Cin, Cout, H, N, T):
    """The shortcut joins windows of three as it joins windows of four: as the two convolutions on their own."""
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    g = gen(9200 + Cin + T)
    x, side = spikes((T, N, Cout, H, H), 0.25, g), spikes((T, N, Cin, 2 * H, 2 * H), 0.25, g)
    w, ws = q(torch.randn(Cout, Cout, 3, 3, generator=g) * 2.0 * (2.0 / (Cout * 9)) ** 0.5, BF16), q(torch.randn(Cout, Cin, 1, 1, generator=g) * (2.0 / Cin) ** 0.5, BF16)
    b, bs = q(torch.randn(Cout, generator=g) * 0.1, BF16), q(torch.randn(Cout, generator=g) * 0.1, BF16)
    sums = [torch.nn.functional.conv2d(side[t], ws, bs, stride=2) for t in range(T)]
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), 1, *LIF, residuals=sums)
    out, v = B.conv_lif_blocked_shortcut(B.from_dense(dev(x, BF16), B.BITS), dev(w, BF16), dev(b, BF16), [1, 1], B.from_dense(dev(side, BF16), B.BITS), dev(ws, BF16),
                                         dev(bs, BF16), [2, 2], LIF, want_v=True)
    assert int(B.last_conv_plan()["variant"]) % 10 == 3
    check(B.to_dense(out), v, ref, what=f"{Cin}->{Cout} {H} T={T}")
