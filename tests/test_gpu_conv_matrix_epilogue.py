"""Dense convolutions of whole tiles with 16-bit spikes on the matrix kernel: spikes leave as bits and the residual arrives through the
wave's stage. Against the CPU oracle for runs of eight and of four pixels, one to four steps per word, several windows, one frame for all
steps, shared tiles of waves, several images per tile, waves without channels and kernels of more than 64 pairs of k-slots."""
import pytest
import torch

from helpers import DEV, LIF, check, dev, gen, q, spikes
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,T,N,dtype,residual,tensor_v,shared", [
    (64, 64, 56, 56, 3, 1, 4, 8, BF16, True, False, False),      # runs of eight
    (64, 128, 28, 28, 3, 1, 3, 5, F16, True, True, False),       # runs of four, an absent step
    (64, 64, 24, 24, 3, 1, 2, 9, BF16, True, True, False),       # words of two steps
    (64, 64, 24, 24, 3, 1, 1, 9, F16, True, True, False),        # one step
    (64, 64, 24, 24, 3, 1, 9, 3, BF16, True, True, False),       # three windows, the last of one step
    (3, 64, 64, 64, 7, 2, 7, 4, F16, True, True, True),          # one frame for seven steps
    (3, 64, 32, 32, 3, 1, 2, 3, BF16, False, False, True),
    (256, 256, 14, 14, 3, 1, 4, 4, BF16, True, True, False),     # eight waves share a tile, runs of four
    (64, 128, 16, 16, 3, 1, 6, 2, F16, True, False, False),
    (256, 512, 2, 2, 3, 1, 4, 9, BF16, True, True, False),       # several images per tile
    (128, 192, 12, 12, 3, 1, 6, 15, F16, True, True, False),     # waves share a tile, those of its last 64 channels of 256 have none
    (64, 64, 24, 24, 7, 1, 4, 2, BF16, False, False, False),     # 98 pairs
    (8, 64, 24, 24, 3, 1, 4, 2, F16, True, False, False),        # one channel group: the last slot of nine is empty
])
def test_whole_tiles_on_the_matrix_kernel(snnf_lib, Cin, Cout, H, W, k, s, T, N, dtype, residual, tensor_v, shared):
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(7800 + Cin + 10 * T + k)
    p = k // 2
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    frame = q(torch.randn(N, Cin, H, W, generator=g), dtype) if shared else None
    xs = [frame if shared else spikes((N, Cin, H, W), 0.25, g) for _ in range(T)]
    w, b = q(torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5, dtype), q(torch.randn(Cout, generator=g) * 0.1, dtype)
    rs = [q(torch.randn(N, Cout, Ho, Wo, generator=g) * 0.3, dtype) for _ in range(T)] if residual else None
    v0 = torch.randn(N, Cout, Ho, Wo, generator=g) * 0.3 if tensor_v else torch.tensor(0.0)
    ref = O.temporal_conv_lif(xs, w, b, v0, (s, s), (p, p), (1, 1), 1, *LIF, residuals=rs)
    one = dev(frame, dtype) if shared else None
    dx, dr, dv = [one if shared else dev(x, dtype) for x in xs], [dev(r, dtype) for r in rs] if residual else None, dev(v0, torch.float32) if tensor_v else None
    packed = CB._packed_weight(dev(w, dtype), dev(b, dtype), dtype)
    sp, v = torch.empty(T, N, Cout, Ho, Wo, device=DEV, dtype=dtype), torch.empty(N, Cout, Ho, Wo, device=DEV)
    _lib.check("conv", snnf_lib.snnf_conv_lif(
        _lib.step_pointers(dx), _lib.step_pointers(dr) if residual else None, T, N, Cin, H, W, _lib.dtype_code(dtype), packed.data_ptr(), Cout, k, k,
        s, s, p, p, _lib.ptr(dv), 0, sp.data_ptr(), int(sp.stride(0)), v.data_ptr(), *LIF, _lib.current_stream(sp.device)))
    plan = CB.last_conv_plan()
    assert plan["kernel"] == "matrix" and int(plan["variant"]) in (21, 22, 24, 31, 34, 32), plan
    check(sp, v, ref, what=f"{Cin}->{Cout} {H}x{W} T={T}")


@pytest.mark.parametrize("Cin,Cout,H,k,s,T,N,residual,moves", [
    (64, 64, 56, 3, 1, 4, 16, False, False),     # seven eighths of one round of full tiles
    (64, 64, 40, 3, 1, 4, 20, True, True),       # tiles of four columns
    (64, 64, 24, 3, 1, 6, 38, True, True),       # less than half a round, two windows
    (128, 256, 28, 3, 2, 8, 5, False, True),
    (64, 128, 56, 3, 2, 4, 16, False, False),
    (64, 128, 56, 1, 2, 4, 16, False, False),
    (16, 64, 40, 3, 1, 4, 2, False, True),       # a single stage: narrow tiles of one wave
    (256, 256, 14, 3, 1, 4, 16, True, True),     # deep: with a residual ...
    (256, 256, 14, 3, 1, 4, 16, False, True),    # ... and without
])
def test_whole_tiles_move_where_they_leave_the_chip_idle(snnf_lib, Cin, Cout, H, k, s, T, N, residual, moves):
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the shapes sit at the edges of 256 compute units")
    g, dtype, p = gen(7900 + Cin + T), BF16, k // 2
    Ho = (H + 2 * p - k) // s + 1
    xs = [dev(spikes((N, Cin, H, H), 0.25, g), dtype) for _ in range(T)]
    w, b = dev(torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5, dtype), dev(torch.randn(Cout, generator=g) * 0.1, dtype)
    rs = [dev(spikes((N, Cout, Ho, Ho), 0.25, g), dtype) for _ in range(T)] if residual else None
    packed, code = CB._packed_weight(w, b, dtype), _lib.dtype_code(dtype)
    need = snnf_lib.snnf_conv_lif_scratch_bytes(T, N, Cin, H, H, code, Cout, k, k, s, s, p, p, 0, int(residual))
    assert (need > 0) == moves
    workspace = torch.empty(max(need, 16), dtype=torch.uint8, device=DEV)
    got = []
    for given in (need, 0):
        sp, v = torch.empty(T, N, Cout, Ho, Ho, device=DEV, dtype=dtype), torch.empty(N, Cout, Ho, Ho, device=DEV)
        _lib.check("conv", snnf_lib.snnf_conv_lif_ws(
            _lib.step_pointers(xs), _lib.step_pointers(rs) if residual else None, T, N, Cin, H, H, code, packed.data_ptr(), Cout, k, k, s, s, p, p,
            None, 0, sp.data_ptr(), int(sp.stride(0)), v.data_ptr(), *LIF, workspace.data_ptr() if given else None, given, _lib.current_stream(sp.device)))
        plan = CB.last_conv_plan()
        assert plan["kernel"] == "matrix" and (plan.get("ran") == "blocked") == (given > 0), plan
        got.append((sp, v))
    rate = float((got[0][0] != got[1][0]).float().mean())       # (sums of the same terms in another order)
    assert rate <= 1e-4 and 0.001 < float(got[0][0].float().mean()) < 0.9, rate
    same = (got[0][0] == got[1][0]).all(0)
    assert torch.allclose(got[0][1][same], got[1][1][same], rtol=1e-3, atol=1e-4)
