"""snnf_conv_lif_ws: layers on dense tensors that are brought into the channel-blocked layout first, against the CPU oracle and
against snnf_conv_lif on the same operands, at the edges of the transposing copy (planes of 8 k pixels, of 4 k, ragged ones, one
pixel; channel counts of a whole and of a part of a group; inputs that start at an odd element) and of the timestep windows."""
import pytest
import torch

from helpers import DEV, LIF, check, dev, gen, q, spikes
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32

CASES = [  # (Cin, Cout, H, W, k, stride, T, N, dtype, residual, tensor v_init, elements the inputs start behind an aligned address)
    (9, 17, 8, 8, 3, 1, 4, 2, BF16, False, False, 0),         # one channel in the second group; 16-byte runs of pixels
    (12, 64, 6, 6, 3, 1, 4, 3, F16, True, True, 0),           # a plane of 4 k pixels
    (20, 40, 5, 7, 3, 1, 3, 2, BF16, True, True, 0),          # 35 pixels: the last run holds three
    (23, 33, 1, 1, 1, 1, 4, 5, BF16, False, True, 0),         # one pixel
    (33, 30, 9, 5, 5, 1, 1, 1, F16, False, False, 0),         # one timestep
    (30, 24, 8, 12, 3, 2, 16, 2, BF16, True, False, 0),       # the longest call, several windows
    (44, 20, 7, 9, 3, 2, 5, 2, BF16, False, True, 1),         # inputs at an odd element, a last window of one step
    (36, 24, 8, 8, 3, 1, 4, 2, BF16, False, False, 4),        # a plane of 8 k pixels at an 8-byte address
    (128, 72, 7, 7, 3, 1, 4, 3, F16, True, True, 0),          # whole groups, the matrix kernel's masked variant
    (300, 64, 3, 3, 3, 1, 6, 1, BF16, True, False, 0),        # K shared by the waves of a workgroup
]


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,T,N,dtype,residual,tensor_v,shift", CASES)
def test_conv_through_the_blocked_layout(snnf_lib, Cin, Cout, H, W, k, s, T, N, dtype, residual, tensor_v, shift):
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(4000 + Cin + Cout + H)
    p = k // 2
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    xs = [q(torch.randn(N, Cin, H, W, generator=g), dtype) if t % 2 else spikes((N, Cin, H, W), 0.25, g) for t in range(T)]
    w, b = q(torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5, dtype), q(torch.randn(Cout, generator=g) * 0.1, dtype)
    rs = [q(torch.randn(N, Cout, Ho, Wo, generator=g) * 0.3, dtype) for _ in range(T)] if residual else None
    v0 = torch.randn(N, Cout, Ho, Wo, generator=g) * 0.3 if tensor_v else torch.tensor(0.0)
    ref = O.temporal_conv_lif(xs, w, b, v0, (s, s), (p, p), (1, 1), 1, *LIF, residuals=rs)
    dx = []
    for x in xs:
        room = torch.zeros(x.numel() + shift, device=DEV, dtype=dtype)
        room[shift:].copy_(x.flatten())
        dx.append(room[shift:].view(x.shape))
    dr = [dev(r, dtype) for r in rs] if residual else None
    dv = dev(v0, F32) if tensor_v else None
    packed = CB._packed_weight(dev(w, dtype), dev(b, dtype), dtype)
    code = _lib.dtype_code(dtype)
    nbytes = snnf_lib.snnf_conv_lif_workspace_bytes(T, N, Cin, H, W, code, Cout, k, k, s, s, p, p, 0, int(residual))
    assert nbytes == T * N * -(-Cin // 8) * H * W * 16
    results, families = {}, {}
    for name, given in (("blocked", nbytes), ("dense", 0), ("short", nbytes - 1)):     # a workspace that is too small is not used
        workspace = torch.full((nbytes,), 255, dtype=torch.uint8, device=DEV)          # NaN patterns
        sp, v = torch.empty(T, N, Cout, Ho, Wo, device=DEV, dtype=dtype), torch.empty(N, Cout, Ho, Wo, device=DEV)
        _lib.check(name, snnf_lib.snnf_conv_lif_ws(
            _lib.step_pointers(dx), _lib.step_pointers(dr) if residual else None, T, N, Cin, H, W, code, packed.data_ptr(), Cout, k, k, s, s, p, p,
            _lib.ptr(dv), 0, sp.data_ptr(), int(sp.stride(0)), v.data_ptr(), *LIF, workspace.data_ptr(), given, _lib.current_stream(sp.device)))
        plan = CB.last_conv_plan()
        assert (plan.get("route") == "c8") == (plan.get("ran") == "blocked") == (name == "blocked"), plan
        check(sp, v, ref, what=f"{name} {Cin}->{Cout} {H}x{W}")
        results[name] = (sp, v)
        families[name] = CB.last_conv_plan()["kernel"]
    assert shift or families["blocked"] == families["dense"], families      # the rule knows which kernel the layer leaves
    assert torch.equal(results["short"][0], results["dense"][0]) and torch.equal(results["short"][1], results["dense"][1])


def test_layers_that_stay_on_the_dense_kernels(snnf_lib):
    bf16, f32 = 1, 0
    asks = snnf_lib.snnf_conv_lif_workspace_bytes
    assert asks(4, 16, 64, 56, 56, bf16, 64, 3, 3, 1, 1, 1, 1, f32, 0) == 0          # whole tiles
    assert asks(4, 32, 128, 28, 28, bf16, 128, 3, 3, 1, 1, 1, 1, f32, 0) == 0        # ... of a deeper layer with many outputs
    assert asks(4, 2, 256, 14, 14, bf16, 256, 3, 3, 1, 1, 1, 1, f32, 0) > 0          # ... of a deep one
    assert asks(4, 16, 128, 56, 56, bf16, 256, 1, 1, 1, 1, 0, 0, f32, 0) == 0        # pointwise
    assert asks(4, 8, 20, 9, 9, f32, 24, 3, 3, 1, 1, 1, 1, f32, 0) == 0              # float32 tensors
    assert asks(1, 8, 20, 9, 9, bf16, 24, 3, 3, 1, 1, 1, 1, bf16, 0) == 0            # 16-bit membrane
    assert asks(17, 8, 20, 9, 9, bf16, 24, 3, 3, 1, 1, 1, 1, f32, 0) == 0            # more timesteps than one launch takes


@pytest.mark.parametrize("Cin,Cout,H,W,N,waves,groups,tiles", [
    (128, 96, 8, 8, 1, "8x1x8", 2, 3),        # few tiles: short stages, so that eight waves share K; tiles of 32 channels
    (128, 40, 8, 8, 1, "8x1x8", 2, 2),        # ... the last of them with 8
    (32, 40, 5, 5, 1, "8x1x2", 2, 2),         # ... two waves each
    (64, 32, 5, 5, 1, "8x1x4", 2, 1),         # ... no more than one tile of channels
    (256, 96, 32, 16, 8, "8x1x8", 4, 2),      # 256 tiles of 64 channels on eight waves: 384 of 32 would be a second round
    (72, 64, 9, 7, 2, "8x1x4", 2, 2),         # nine channel groups: the last stage holds one
    (128, 64, 32, 40, 13, "8x1x2", 4, 1),     # 520 tiles: four waves each would be a second round
    (128, 64, 32, 40, 26, "8x1x1", 4, 1),     # 1040 tiles: two waves each would be a second round
])
def test_waves_that_share_a_tile(snnf_lib, Cin, Cout, H, W, N, waves, groups, tiles):
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the shapes sit at the edges of 256 compute units")
    g = gen(4500 + N)
    x = torch.stack([spikes((N, Cin, H, W), 0.25, g) for _ in range(4)])
    w, b = q(torch.randn(Cout, Cin, 3, 3, generator=g) * 2.0 * (2.0 / (Cin * 9)) ** 0.5, BF16), q(torch.randn(Cout, generator=g) * 0.1, BF16)
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), 1, *LIF)
    out, v = B.conv_lif_blocked(B.from_dense(dev(x, BF16), B.BITS), dev(w, BF16), dev(b, BF16), [1, 1], [1, 1], LIF, out_layout=B.BITS, want_v=True)
    plan = B.last_conv_plan()
    assert (plan["waves"], int(plan["stage_chunks"]), int(plan["oc_tiles"])) == (waves, groups, tiles), plan
    assert plan["oc_tiles"] == -(-Cout // plan["oc_tile"])
    check(B.to_dense(out), v, ref, what=f"{Cin}->{Cout} {H}x{W} x {N}")


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,T,N,residual", [(128, 72, 7, 7, 3, 1, 4, 3, True), (256, 40, 6, 7, 3, 2, 5, 2, False), (480, 24, 9, 9, 1, 2, 1, 2, False)])
def test_convolution_without_a_neuron(snnf_lib, Cin, Cout, H, W, k, s, T, N, residual):
    """Against float64 sums rounded once to bf16: half a unit in the last place (2^-8 relative) and the float32 sums' own error."""
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(4700 + Cin)
    p = k // 2
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    xs = [q(torch.randn(N, Cin, H, W, generator=g), BF16) for _ in range(T)]
    w, b = q(torch.randn(Cout, Cin, k, k, generator=g) * (1.0 / (Cin * k * k)) ** 0.5, BF16), q(torch.randn(Cout, generator=g) * 0.1, BF16)
    rs = [q(torch.randn(N, Cout, Ho, Wo, generator=g), BF16) for _ in range(T)] if residual else None
    out = CB.run_hip_temporal_conv_bias([dev(x, BF16) for x in xs], dev(w, BF16), dev(b, BF16), [s, s], [p, p],
                                        [dev(r, BF16) for r in rs] if residual else None)
    want = k == 3 or T > 2
    assert (CB.last_conv_plan().get("route") == "c8") == want, CB.last_conv_plan()
    ref = torch.stack([torch.nn.functional.conv2d(x.double(), w.double(), b.double(), s, p) + (rs[t].double() if residual else 0) for t, x in enumerate(xs)])
    assert torch.all((out.double().cpu() - ref).abs() <= ref.abs() * 2.0 ** -8 + 1e-4)


@pytest.mark.parametrize("Cin,Cout,H,W,N,grid", [(16, 64, 8, 8, 3, 6), (16, 64, 40, 40, 46, 256), (16, 64, 56, 56, 16, 196)])
def test_tiles_spread_over_compute_units(snnf_lib, Cin, Cout, H, W, N, grid):
    """Six tiles on six workgroups; 2300 tiles in two rounds of 256 workgroups (144 full ones would leave 112 units idle); 1568 in
    one round of 196 full workgroups."""
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the shapes sit at the edges of 256 compute units")
    g = gen(4800 + N)
    x = torch.stack([spikes((N, Cin, H, W), 0.25, g) for _ in range(4)])
    w, b = q(torch.randn(Cout, Cin, 3, 3, generator=g) * 2.0 * (2.0 / (Cin * 9)) ** 0.5, BF16), q(torch.randn(Cout, generator=g) * 0.1, BF16)
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), 1, *LIF)
    out, v = B.conv_lif_blocked(B.from_dense(dev(x, BF16), B.BITS), dev(w, BF16), dev(b, BF16), [1, 1], [1, 1], LIF, out_layout=B.BITS, want_v=True)
    assert int(B.last_conv_plan()["grid"]) == grid, B.last_conv_plan()
    check(B.to_dense(out), v, ref, what=f"{Cin}->{Cout} {H}x{W} x {N}")


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,N,dtype,layout,tile", [
    (32, 512, 2, 2, 5, 1, 123, BF16, "bits", "4x2x2"),      # the halos of eight planes of 6 x 6 don't fit, those of four do
    (32, 512, 4, 4, 3, 2, 125, BF16, "bits", "4x2x2"),      # ... of 5 x 5
    (64, 512, 8, 8, 3, 2, 66, F16, "c8", "1x4x4"),          # two planes of 9 x 9
    (32, 64, 2, 2, 5, 1, 257, F16, "nchw", "4x2x2"),        # ... and dense tensors around, as a call of two launches
    (32, 64, 4, 4, 5, 2, 64, BF16, "bits", "1x2x1"),        # 256 pixels: parts of planes
    (32, 64, 4, 4, 5, 2, 65, BF16, "bits", "2x2x2"),        # 260: whole ones
])
def test_whole_planes_whose_halos_do_not_fit(snnf_lib, Cin, Cout, H, W, k, s, N, dtype, layout, tile):
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the shapes sit at the edges of 256 compute units")
    g = gen(5000 + N)
    p = k // 2
    x = torch.stack([spikes((N, Cin, H, W), 0.25, g) for _ in range(4)])
    w, b = q(torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5, dtype), q(torch.randn(Cout, generator=g) * 0.1, dtype)
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (s, s), (p, p), (1, 1), 1, *LIF)
    if layout == "nchw":
        dx, Ho, Wo = [dev(t, dtype) for t in x], (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
        from triton_snn_fusion_amd import _lib
        need = snnf_lib.snnf_conv_lif_scratch_bytes(4, N, Cin, H, W, _lib.dtype_code(dtype), Cout, k, k, s, s, p, p, 0, 0)
        assert need > 0
        workspace, packed = torch.empty(need, dtype=torch.uint8, device=DEV), CB._packed_weight(dev(w, dtype), dev(b, dtype), dtype)
        sp, v = torch.empty(4, N, Cout, Ho, Wo, device=DEV, dtype=dtype), torch.empty(N, Cout, Ho, Wo, device=DEV)
        _lib.check("snnf_conv_lif_ws", snnf_lib.snnf_conv_lif_ws(
            _lib.step_pointers(dx), None, 4, N, Cin, H, W, _lib.dtype_code(dtype), packed.data_ptr(), Cout, k, k, s, s, p, p, None, 0,
            sp.data_ptr(), int(sp.stride(0)), v.data_ptr(), *LIF, workspace.data_ptr(), need, _lib.current_stream(sp.device)))
    else:
        layout = {"bits": B.BITS, "c8": B.C8}[layout]
        out, v = B.conv_lif_blocked(B.from_dense(dev(x, dtype), layout), dev(w, dtype), dev(b, dtype), [s, s], [p, p], LIF, out_layout=layout, want_v=True)
        sp = B.to_dense(out)
    assert CB.last_conv_plan()["tile"] == tile, CB.last_conv_plan()
    check(sp, v, ref, what=f"{Cin}->{Cout} {k}x{k}/{s} {H}x{W} x {N}")


@pytest.mark.parametrize("T,out", [(1, "bits"), (2, "bits"), (1, "c8"), (2, "nchw")])
def test_narrow_tiles_of_short_windows(snnf_lib, T, out):
    """One and two timesteps on tiles of 32 channels, straight-line and general epilogue, a last tile of 8 channels."""
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    layout = {"bits": B.BITS, "c8": B.C8, "nchw": B.NCHW}[out]
    g = gen(4900 + T)
    x = torch.stack([spikes((2, 128, 9, 7), 0.25, g) for _ in range(T)])
    w, b = q(torch.randn(40, 128, 3, 3, generator=g) * 2.0 * (2.0 / 1152) ** 0.5, BF16), q(torch.randn(40, generator=g) * 0.1, BF16)
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), 1, *LIF)
    got, v = B.conv_lif_blocked(B.from_dense(dev(x, BF16), B.BITS), dev(w, BF16), dev(b, BF16), [1, 1], [1, 1], LIF, out_layout=layout, want_v=True)
    assert int(B.last_conv_plan()["oc_tiles"]) == 2, B.last_conv_plan()
    check(B.to_dense(got), v, ref, what=f"T={T} {out}")


def test_one_frame_for_all_timesteps_takes_no_scratch_memory(hip_ops):
    """The operator, on its first call and once it is known, and the neuron-free convolution allocate their outputs and nothing else;
    with a frame per timestep the scratch of the blocked route comes on top."""
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    S = torch.ops.snn_custom
    g = gen(4950)
    frames = [dev(spikes((8, 72, 33, 33), 0.25, g), BF16) for _ in range(4)]
    w, b = dev(torch.randn(40, 72, 3, 3, generator=g), BF16), dev(torch.randn(40, generator=g), BF16)
    zero = torch.zeros((), device=DEV)
    operator = lambda xs: S.fused_temporal_conv_lif_state(xs, w, b, zero, [1, 1], [1, 1], [1, 1], 1, *LIF, False)
    neuron_free = lambda xs: CB.run_hip_temporal_conv_bias(xs, w, b, [1, 1], [1, 1])
    scratch = 4 * 8 * 9 * 33 * 33 * 16
    for call, outputs in ((operator, (4 * 2 + 4) * 8 * 40 * 33 * 33), (neuron_free, 4 * 2 * 8 * 40 * 33 * 33)):
        call(frames)                                            # packs the weight
        for xs, extra in (([frames[0]] * 4, 0), (frames, scratch)):
            for _ in range(3):
                torch.cuda.reset_peak_memory_stats()
                before = torch.cuda.memory_stats()["requested_bytes.all.current"]
                out = call(xs)
                assert torch.cuda.memory_stats()["requested_bytes.all.peak"] - before == outputs + extra
                del out
