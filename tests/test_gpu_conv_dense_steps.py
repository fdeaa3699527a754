"""Dense convolutions whose kernel reads the frames of the timesteps itself, without a copy in another layout: against the CPU oracle at the edges of pairs of pixels,
rows and channel groups, where an infinity or NaN beside the image, the channels or the batch must not be met, and the general path for other neurons."""
import pytest
import torch

from helpers import DEV, LIF, check, dev, gen, q, spikes
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
SOFT = (1.0, -1.0, 2.0)


def _run(xs, rs, w, b, zero, s, p, lif):
    S = torch.ops.snn_custom
    args = (w, b, zero, [s, s], [p, p], [1, 1], 1, *lif, False)
    return S.fused_temporal_conv_lif_state(xs, *args) if rs is None else S.fused_temporal_conv_add_lif_state(xs, rs, *args)


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,N,T,dtype,residual,lif,route", [
    (64, 64, 32, 32, 3, 1, 8, 4, BF16, False, LIF, "frames"),     # whole groups, four waves a tile
    (20, 33, 13, 17, 3, 1, 12, 4, F16, True, LIF, "frames"),       # odd rows and single channels, in and out
    (72, 104, 27, 35, 3, 1, 2, 6, F16, True, LIF, "frames"),       # windows of three
    (64, 64, 24, 24, 3, 1, 4, 5, BF16, True, LIF, "frames"),       # one window
    (40, 48, 9, 9, 5, 1, 20, 2, BF16, False, LIF, "frames"),
    (48, 24, 23, 21, 3, 2, 16, 3, BF16, False, LIF, "frames"),     # stride 2: pairs half of which no window reads
    (30, 18, 5, 31, 1, 1, 40, 8, BF16, True, LIF, "frames"),       # 1x1, odd rows, two windows
    (128, 96, 3, 64, 3, 1, 14, 1, F16, False, LIF, "frames"),      # one timestep
    (24, 40, 64, 2, 3, 1, 30, 4, BF16, False, LIF, "frames"),      # rows of two pixels
    (24, 40, 64, 1, 3, 1, 40, 4, BF16, False, LIF, "c8"),         # of one: no pairs
    (16, 64, 40, 40, 3, 1, 12, 4, BF16, True, LIF, None),         # a wave a tile
    (32, 64, 12, 12, 3, 1, 1, 4, BF16, False, SOFT, "frames"),    # few pixels, any neuron
    (20, 30, 9, 7, 3, 1, 2, 8, F16, True, LIF, "frames"),         # two windows, single channels
    (40, 64, 14, 13, 5, 1, 1, 2, BF16, False, LIF, "frames"),
    (72, 40, 11, 1, 3, 1, 3, 4, BF16, True, LIF, "frames"),       # rows of one pixel
    (96, 104, 33, 31, 1, 1, 4, 2, BF16, True, LIF, "frames"),     # 1x1 of two timesteps
    (96, 104, 33, 31, 1, 1, 4, 2, BF16, True, SOFT, None),        # and on the dense kernels for another neuron
    (136, 32, 68, 11, 1, 1, 9, 1, F16, False, LIF, "frames"),
    (512, 64, 7, 7, 3, 1, 1, 4, BF16, False, LIF, "c8"),          # too many channels for a workgroup's loads
    (64, 64, 32, 32, 3, 1, 8, 4, BF16, False, SOFT, "c8"),        # another neuron: the copy
])
def test_against_the_oracle(hip_ops, snnf_lib, Cin, Cout, H, W, k, s, N, T, dtype, residual, lif, route):
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(9300 + Cin + Cout + T)
    p = k // 2
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    x = q(torch.randn(T, N, Cin, H, W, generator=g), dtype)      # any values
    w, b = q(torch.randn(Cout, Cin, k, k, generator=g) * (2.0 / (Cin * k * k)) ** 0.5, dtype), q(torch.randn(Cout, generator=g) * 0.1, dtype)
    rs = torch.stack([spikes((N, Cout, Ho, Wo), 0.25, g) for _ in range(T)]) if residual else None
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (s, s), (p, p), (1, 1), 1, *lif, residuals=list(rs) if residual else None)
    # Every frame lies between infinities, one element off an address of four bytes.
    frame = N * Cin * H * W
    room = torch.full((T, frame + 2 + frame % 2), float("inf"), dtype=dtype, device=DEV)
    xs = [room[t, 1:1 + frame].view(N, Cin, H, W) for t in range(T)]
    for t in range(T):
        xs[t].copy_(x[t])
    sp, v = _run(xs, None if rs is None else [dev(t, dtype) for t in rs], dev(w, dtype), dev(b, dtype), torch.zeros((), device=DEV), s, p, lif)
    plan = CB.last_conv_plan()
    if route is not None and torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert plan.get("reads", plan.get("route")) == route, plan
    check(sp, v, ref, what=f"{Cin}->{Cout} {H}x{W} T={T}", max_rate=1e-3)


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,N,T,residual,low", [
    (64, 64, 32, 32, 3, 1, 8, 4, False, "none"),          # spikes: no low terms
    (64, 64, 32, 32, 3, 1, 8, 4, False, "all"),
    (72, 24, 14, 14, 3, 1, 3, 4, True, "one"),            # five stages on four waves, a low term in the last one alone
    (88, 40, 20, 19, 3, 1, 4, 3, False, "one"),           # six on four, odd rows
    (20, 33, 13, 17, 3, 1, 6, 6, True, "all"),            # single channels, windows of three
    (168, 24, 9, 9, 3, 2, 6, 2, False, "all"),            # eight waves, stride 2
    (30, 18, 5, 31, 1, 1, 20, 1, True, "one"),            # 1x1, one timestep
    (16, 24, 30, 31, 3, 1, 20, 5, False, "all"),          # one stage: a wave a tile
])
def test_fp32_terms_against_the_oracle(hip_ops, snnf_lib, Cin, Cout, H, W, k, s, N, T, residual, low):
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(9350 + Cin + Cout + T)
    p = k // 2
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    x = torch.randn(T, N, Cin, H, W, generator=g) if low == "all" else spikes((T, N, Cin, H, W), 0.3, g)
    if low == "one":
        x[T - 1, N - 1, Cin - 1, H // 2, W - 1] = 1.0 + 2.0 ** -10       # (a low term that a bf16 sum over the window shows)
    w, b = torch.randn(Cout, Cin, k, k, generator=g) * (2.0 / (Cin * k * k)) ** 0.5, torch.randn(Cout, generator=g) * 0.1
    rs = torch.stack([spikes((N, Cout, Ho, Wo), 0.25, g) for _ in range(T)]) if residual else None
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (s, s), (p, p), (1, 1), 1, *LIF, residuals=list(rs) if residual else None)
    frame = N * Cin * H * W
    room = torch.full((T, frame + 2), float("inf"), device=DEV)
    xs = [room[t, 1:1 + frame].view(N, Cin, H, W) for t in range(T)]
    for t in range(T):
        xs[t].copy_(x[t])
    sp, v = _run(xs, None if rs is None else [dev(t, F32) for t in rs], dev(w, F32), dev(b, F32), torch.zeros((), device=DEV), s, p, LIF)
    plan = CB.last_conv_plan()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert plan.get("reads") == "frames", plan
    check(sp, v, ref, what=f"{Cin}->{Cout} {H}x{W} T={T}", max_rate=1e-3)
    if low == "one":      # the low term's own share: the call without it, on the neurons that have the same spikes
        xs[T - 1][N - 1, Cin - 1, H // 2, W - 1] = 1.0
        sp1, v1 = _run(xs, None if rs is None else [dev(t, F32) for t in rs], dev(w, F32), dev(b, F32), torch.zeros((), device=DEV), s, p, LIF)
        same = (sp == sp1).all(0) & (sp[-1] == 0)
        changed = ((v - v1) != 0) & same
        assert int(changed.sum()) > 0 and int(changed[:N - 1].sum()) == 0


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,N,T,dtype", [
    (264, 101, 67, 67, 3, 1, 1, 4, BF16),         # many loads to a tile
    (456, 32, 16, 17, 1, 1, 8, 8, BF16),          # 1x1 in columns of two pixels
    (116, 72, 34, 27, 7, 2, 25, 1, BF16),         # two waves a tile instead of four, for its wider halo
    (328, 40, 10, 53, 1, 1, 11, 6, F32),
])
def test_layers_that_the_copy_is_faster_for(hip_ops, snnf_lib, Cin, Cout, H, W, k, s, N, T, dtype):
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(9370 + Cin)
    p = k // 2
    x, b = [spikes((N, Cin, H, W), 0.2, g) for _ in range(T)], torch.randint(-16, 17, (Cout,), generator=g) / 64.0
    w = torch.randint(-64, 65, (Cout, Cin, k, k), generator=g) / 512.0      # (sums that are exact in any order)
    sp, v = _run([dev(t, dtype) for t in x], None, dev(w, dtype), dev(b, dtype), torch.zeros((), device=DEV), s, p, LIF)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        plan = CB.last_conv_plan()
        assert plan.get("reads") is None and plan.get("route") == "c8", plan
    ref = O.temporal_conv_lif(x, w, b, torch.tensor(0.0), (s, s), (p, p), (1, 1), 1, *LIF)
    assert torch.equal(sp.float().cpu(), ref[0]) and 0.0 < float(ref[0].mean()) < 1.0
    check(sp, v, ref, what=f"{Cin}->{Cout} {H}x{W} T={T}")


@pytest.mark.parametrize("Cin,Cout,H,W,N,T,residual,dtype,route", [
    (168, 104, 110, 58, 8, 1, True, BF16, None),      # no copy to fall back to: the dense kernel
    (456, 86, 32, 83, 6, 2, False, F16, None),
    (112, 24, 16, 57, 31, 4, False, BF16, "c8"),
    (112, 24, 16, 57, 31, 4, False, F32, "c8"),
])
def test_large_frames_in_narrow_patches_of_1x1(hip_ops, snnf_lib, Cin, Cout, H, W, N, T, residual, dtype, route):
    """Every tile of two or four columns would fetch whole lines, gone from the L2 caches before its neighbour's turn."""
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(9375 + Cin)
    x, b = [spikes((N, Cin, H, W), 0.2, g) for _ in range(T)], torch.randint(-16, 17, (Cout,), generator=g) / 64.0
    rs = [spikes((N, Cout, H, W), 0.2, g) for _ in range(T)] if residual else None
    w = torch.randint(-64, 65, (Cout, Cin, 1, 1), generator=g) / 128.0      # (sums that are exact in any order)
    sp, v = _run([dev(t, dtype) for t in x], [dev(t, dtype) for t in rs] if residual else None, dev(w, dtype), dev(b, dtype), torch.zeros((), device=DEV), 1, 0, LIF)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        plan = CB.last_conv_plan()
        assert plan.get("reads") is None and plan.get("route") == route, plan
    ref = O.temporal_conv_lif(x, w, b, torch.tensor(0.0), (1, 1), (0, 0), (1, 1), 1, *LIF, residuals=rs)
    assert torch.equal(sp.float().cpu(), ref[0]) and 0.0 < float(ref[0].mean()) < 1.0
    check(sp, v, ref, what=f"{Cin}->{Cout} {H}x{W} T={T}")


@pytest.mark.parametrize("Cin,Cout,H,k,s,N,T", [
    (27, 328, 15, 7, 2, 5, 4),       # whose frames would take two windows where the copy takes one
    (72, 104, 27, 3, 1, 2, 6),       # two of each
    (64, 64, 24, 3, 1, 4, 5),        # one of six
    (48, 40, 20, 5, 1, 6, 3),
])
def test_scratch_memory_is_not_left(hip_ops, snnf_lib, Cin, Cout, H, k, s, N, T):
    """A 16-bit membrane passes from window to window in the scratch memory that the query asks for: what lies behind it stays as it was."""
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(9380 + Cin)
    p, code = k // 2, _lib.dtype_code(F16)
    Ho = (H + 2 * p - k) // s + 1
    x = [spikes((N, Cin, H, H), 0.25, g) for _ in range(T)]
    xs = [dev(t, F16) for t in x]
    w, b = q(torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5, F16), q(torch.randn(Cout, generator=g) * 0.1, F16)
    packed = CB._packed_weight(dev(w, F16), dev(b, F16), F16)
    need = snnf_lib.snnf_conv_lif_scratch_bytes(T, N, Cin, H, H, code, Cout, k, k, s, s, p, p, code, 0)
    room = torch.full((need + N * Cout * Ho * Ho * 4 + 4096,), 171, dtype=torch.uint8, device=DEV)      # (a whole fp32 membrane behind it)
    sp, v = torch.empty(T, N, Cout, Ho, Ho, device=DEV, dtype=F16), torch.empty(N, Cout, Ho, Ho, device=DEV, dtype=F16)
    _lib.check("ws", snnf_lib.snnf_conv_lif_ws(_lib.step_pointers(xs), None, T, N, Cin, H, H, code, packed.data_ptr(), Cout, k, k, s, s, p, p, None, code,
                                               sp.data_ptr(), int(sp.stride(0)), v.data_ptr(), *LIF, room.data_ptr(), need, _lib.current_stream(sp.device)))
    assert CB.last_conv_plan().get("ran") == "blocked"
    assert int((room[need:] != 171).sum()) == 0
    check(sp, v, O.temporal_conv_lif(x, w, b, torch.tensor(0.0), (s, s), (p, p), (1, 1), 1, *LIF), v_dtype=F16)


@pytest.mark.parametrize("T,v_dtype", [(1, F32), (2, F32), (2, BF16)])
def test_1x1_of_up_to_two_timesteps_needs_no_copy(hip_ops, snnf_lib, T, v_dtype):
    """Layers that are on this route only where the kernel reads their frames ask for a token, not for the room of a copy, and leave it as it is."""
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(9385)
    N, Cin, Cout, H, W, code = 9, 144, 104, 10, 54, _lib.dtype_code(BF16)
    x = [spikes((N, Cin, H, W), 0.25, g) for _ in range(T)]
    xs = [dev(t, BF16) for t in x]
    w, b = q(torch.randn(Cout, Cin, 1, 1, generator=g) * 2.0 * (2.0 / Cin) ** 0.5, BF16), q(torch.randn(Cout, generator=g) * 0.1, BF16)
    packed = CB._packed_weight(dev(w, BF16), dev(b, BF16), BF16)
    need = snnf_lib.snnf_conv_lif_scratch_bytes(T, N, Cin, H, W, code, Cout, 1, 1, 1, 1, 0, 0, _lib.dtype_code(v_dtype), 0)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert need == 16 * T
    room = torch.full((max(need, 16) + 4096,), 171, dtype=torch.uint8, device=DEV)
    sp, v = torch.empty(T, N, Cout, H, W, device=DEV, dtype=BF16), torch.empty(N, Cout, H, W, device=DEV, dtype=v_dtype)
    _lib.check("ws", snnf_lib.snnf_conv_lif_ws(_lib.step_pointers(xs), None, T, N, Cin, H, W, code, packed.data_ptr(), Cout, 1, 1, 1, 1, 0, 0, None, _lib.dtype_code(v_dtype),
                                               sp.data_ptr(), int(sp.stride(0)), v.data_ptr(), *LIF, room.data_ptr(), need, _lib.current_stream(sp.device)))
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert CB.last_conv_plan().get("reads") == "frames"
    assert bool((room == 171).all())
    check(sp, v, O.temporal_conv_lif(x, w, b, torch.tensor(0.0), (1, 1), (0, 0), (1, 1), 1, *LIF), v_dtype=v_dtype)


@pytest.mark.parametrize("N,H", [(8, 32), (1, 12)])      # tiles, few pixels
def test_spikes_over_the_inputs(hip_ops, snnf_lib, N, H):
    """Inputs that the spikes are written over are copied first."""
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(9395)
    T, C, code = 4, 32, _lib.dtype_code(BF16)
    x = torch.stack([spikes((N, C, H, H), 0.25, g) for _ in range(T)])
    w, b = dev(torch.randn(C, C, 3, 3, generator=g) * 0.2, BF16), dev(torch.randn(C, generator=g) * 0.1, BF16)
    packed = CB._packed_weight(w, b, BF16)
    need = snnf_lib.snnf_conv_lif_scratch_bytes(T, N, C, H, H, code, C, 3, 3, 1, 1, 1, 1, 0, 0)
    room, got = torch.empty(need, dtype=torch.uint8, device=DEV), []
    for over in (False, True):
        xs = dev(x, BF16)
        sp, v = xs if over else torch.empty_like(xs), torch.empty(N, C, H, H, device=DEV)
        _lib.check("ws", snnf_lib.snnf_conv_lif_ws(_lib.step_pointers(list(xs)), None, T, N, C, H, H, code, packed.data_ptr(), C, 3, 3, 1, 1, 1, 1, None, 0, sp.data_ptr(),
                                                   int(sp.stride(0)), v.data_ptr(), *LIF, room.data_ptr(), need, _lib.current_stream(sp.device)))
        got.append((sp.clone(), v))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and 0 < float(got[0][0].float().mean()) < 1


@pytest.mark.parametrize("N,H", [(8, 32), (1, 12)])      # tiles, few pixels
def test_inputs_right_behind_a_16bit_membrane_are_no_overlap(hip_ops, snnf_lib, N, H):
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(9396)
    T, C, code = 4, 32, _lib.dtype_code(BF16)
    n = N * C * H * H
    x = torch.stack([spikes((N, C, H, H), 0.25, g) for _ in range(T)])
    w, b = q(torch.randn(C, C, 3, 3, generator=g) * 0.2, BF16), q(torch.randn(C, generator=g) * 0.1, BF16)
    packed = CB._packed_weight(dev(w, BF16), dev(b, BF16), BF16)
    need = snnf_lib.snnf_conv_lif_scratch_bytes(T, N, C, H, H, code, C, 3, 3, 1, 1, 1, 1, code, 0)
    both, room = torch.empty((T + 1) * n, device=DEV, dtype=BF16), torch.empty(need, dtype=torch.uint8, device=DEV)
    v, xs = both[:n].view(N, C, H, H), both[n:].view(T, N, C, H, H)
    xs.copy_(x)
    sp = torch.empty(T, N, C, H, H, device=DEV, dtype=BF16)
    _lib.check("ws", snnf_lib.snnf_conv_lif_ws(_lib.step_pointers(list(xs)), None, T, N, C, H, H, code, packed.data_ptr(), C, 3, 3, 1, 1, 1, 1, None, code, sp.data_ptr(),
                                               int(sp.stride(0)), v.data_ptr(), *LIF, room.data_ptr(), need, _lib.current_stream(sp.device)))
    if torch.cuda.get_device_properties(0).multi_processor_count == 256 and N > 1:      # (the plan of few pixels names its frames either way)
        assert CB.last_conv_plan().get("reads") == "frames"
    check(sp, v, O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), 1, *LIF), v_dtype=BF16)


def test_infinities_stay_in_their_windows(hip_ops, snnf_lib):
    """An infinity in the last channel of an image reaches its own windows and no neighbour's: pixels outside the image and channels beyond the last are zeros."""
    g = gen(9390)
    T, N, C, H, W = 4, 10, 20, 11, 13
    x = spikes((T, N, C, H, W), 0.3, g)
    w, b = q(torch.randn(24, C, 3, 3, generator=g) * 0.2, BF16), q(torch.randn(24, generator=g) * 0.1, BF16)
    clean, _ = _run([dev(t, BF16) for t in x], None, dev(w, BF16), dev(b, BF16), torch.zeros((), device=DEV), 1, 1, LIF)
    bad = x.clone()
    bad[:, 4, C - 1, H - 1, W - 1] = float("nan")
    got, _ = _run([dev(t, BF16) for t in bad], None, dev(w, BF16), dev(b, BF16), torch.zeros((), device=DEV), 1, 1, LIF)
    met = torch.zeros(T, N, 24, H, W, dtype=torch.bool)
    met[:, 4, :, H - 2:, W - 2:] = True
    assert torch.equal(got.cpu()[~met], clean.cpu()[~met])
