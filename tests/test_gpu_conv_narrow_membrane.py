"""Dense convolutions with a 16-bit membrane on the blocked kernel: held in fp32 over all windows and rounded once, as the same call with
an fp32 membrane rounded afterwards; through the library's entry point and through the operator, from zeros and from a tensor."""
import pytest
import torch

from helpers import DEV, LIF, dev, gen, q, spikes

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
SOFT = (1.0, -1.0, 2.0)


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,T,N,dtype,residual,tensor_v,lif", [
    (72, 104, 27, 35, 3, 1, 6, 2, F16, True, False, LIF),       # two windows
    (72, 40, 9, 9, 3, 1, 4, 2, BF16, False, True, LIF),         # one window: nothing is carried
    (20, 33, 5, 7, 3, 2, 9, 2, BF16, True, True, LIF),          # three windows, single channels masked
    (64, 64, 24, 24, 3, 1, 16, 4, BF16, False, True, SOFT),     # four, the general epilogue
    (128, 72, 7, 7, 3, 1, 1, 3, F16, True, True, LIF),          # one step
    (40, 26, 13, 13, 1, 1, 5, 2, BF16, True, False, LIF),       # pointwise
])
def test_narrow_membrane_is_rounded_once(hip_ops, snnf_lib, Cin, Cout, H, W, k, s, T, N, dtype, residual, tensor_v, lif):
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g = gen(7600 + Cin + T)
    p = k // 2
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    xs = [dev(spikes((N, Cin, H, W), 0.25, g), dtype) for _ in range(T)]
    w, b = dev(torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5, dtype), dev(torch.randn(Cout, generator=g) * 0.1, dtype)
    rs = [dev(spikes((N, Cout, Ho, Wo), 0.25, g), dtype) for _ in range(T)] if residual else None
    v0 = dev(torch.randn(N, Cout, Ho, Wo, generator=g) * 0.3, dtype) if tensor_v else None
    packed, code = CB._packed_weight(w, b, dtype), _lib.dtype_code(dtype)
    got = {}
    for v_dtype in (dtype, F32):
        need = snnf_lib.snnf_conv_lif_scratch_bytes(T, N, Cin, H, W, code, Cout, k, k, s, s, p, p, _lib.dtype_code(v_dtype), int(residual))
        carried = N * Cout * Ho * Wo * 4 if v_dtype == dtype and T > 4 else 0
        assert need == T * N * -(-Cin // 8) * H * W * 16 + carried
        workspace = torch.full((need,), 255, dtype=torch.uint8, device=DEV)
        sp, v = torch.empty(T, N, Cout, Ho, Wo, device=DEV, dtype=dtype), torch.empty(N, Cout, Ho, Wo, device=DEV, dtype=v_dtype)
        start = None if v0 is None else v0.to(v_dtype)
        _lib.check("ws", snnf_lib.snnf_conv_lif_ws(
            _lib.step_pointers(xs), _lib.step_pointers(rs) if residual else None, T, N, Cin, H, W, code, packed.data_ptr(), Cout, k, k, s, s, p, p,
            _lib.ptr(start), _lib.dtype_code(v_dtype), sp.data_ptr(), int(sp.stride(0)), v.data_ptr(), *lif, workspace.data_ptr(), need,
            _lib.current_stream(sp.device)))
        assert CB.last_conv_plan().get("ran") == "blocked", CB.last_conv_plan()
        got[v_dtype] = (sp, v)
    assert torch.equal(got[dtype][0], got[F32][0]) and torch.equal(got[dtype][1], got[F32][1].to(dtype))
    assert 0.001 < float(got[F32][0].float().mean()) < 0.9
    S = torch.ops.snn_custom
    geometry = ([s, s], [p, p], [1, 1], 1)
    for _ in range(3):                                          # the Python implementation, then the native one
        start = torch.zeros(()) if v0 is None else v0
        sp, v = (S.fused_temporal_conv_add_lif_state(xs, rs, w, b, start, *geometry, *lif, False) if residual
                 else S.fused_temporal_conv_lif_state(xs, w, b, start, *geometry, *lif, False))
        assert v.dtype == dtype and CB.last_conv_plan().get("ran") == "blocked"
        assert torch.equal(sp, got[dtype][0]) and torch.equal(v, got[dtype][1])
