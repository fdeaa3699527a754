"""Depthwise 3x3 of stride 1 on 16-bit rows that are no whole 16-byte vectors, or start between them, against the oracle: strips that overlap the one before, first and last rows and
planes beside infinities, membranes of either type, and in place.

Weights, biases and inputs are fixed-point numbers whose sums of nine are exact in float32: spikes and membranes are the oracle's bit for bit."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import DEV, LIF, dev, gen, q, spikes
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
SOFT = (1.0, -1.0, 3.0)


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("N,C,H,W,T,residual,v_dtype,start,lif", [
    (1, 2, 1, 9, 1, False, F32, False, LIF),          # one row; the second strip is one pixel
    (2, 3, 2, 15, 2, True, F32, False, LIF),
    (3, 5, 7, 8, 3, False, F32, True, LIF),           # whole vectors that start between them
    (2, 3, 11, 13, 2, True, None, True, LIF),         # a membrane of the activations' type
    (2, 70, 40, 31, 5, False, F32, False, LIF),       # odd rows of several steps, in many strips
    (1, 230, 30, 17, 4, True, None, True, LIF),
    (1, 70, 17, 17, 5, False, F32, False, LIF),       # and in few: in LDS
    (2, 6, 20, 20, 2, True, F32, False, LIF),         # rows of a multiple of four
    (1, 9, 9, 30, 20, False, F32, False, LIF),        # a second launch, which goes on in place
    (2, 3, 5, 7, 3, True, F32, False, LIF),           # shorter than a strip
    (1, 4, 9, 31, 2, True, F32, True, SOFT),
])
def test_rows_that_start_and_end_anywhere(hip_ops, snnf_lib, N, C, H, W, T, residual, v_dtype, start, lif, dtype):
    from triton_snn_fusion_amd import _lib
    g = gen(5200 + C + W + T)
    v_dtype = dtype if v_dtype is None else v_dtype
    w, b = torch.randint(-64, 65, (C, 1, 3, 3), generator=g) / 64.0, torch.randint(-16, 17, (C,), generator=g) / 64.0
    x = torch.randint(-8, 9, (T, N, C, H, W), generator=g) / 4.0
    rs = torch.stack([spikes((N, C, H, W), 0.3, g) for _ in range(T)]) if residual else None
    v0 = q(torch.randn(N, C, H, W, generator=g) * 0.3, v_dtype) if start else torch.tensor(0.0)
    ref = O.temporal_conv_lif(list(x), w, b, v0, (1, 1), (1, 1), (1, 1), C, *lif, residuals=list(rs) if residual else None)
    n = N * C * H * W

    def between(t, dt):        # one element off a whole vector, infinities on both sides
        room = torch.full((n + 16,), float("inf"), dtype=dt, device=DEV)
        room[1:1 + n].copy_(t.flatten())
        return room[1:1 + n].view(N, C, H, W)

    xs = [between(t, dtype) for t in x]
    rp = [between(t, dtype) for t in rs] if residual else None
    dw, db = dev(w, dtype), dev(b, dtype)
    got = {}
    for in_place in ((False, True) if start else (False,)):
        room = torch.full((T * n + 16,), 7.0, dtype=dtype, device=DEV)
        sp, v = room[1:1 + T * n].view(T, N, C, H, W), between(torch.zeros(N, C, H, W), v_dtype)
        if in_place:
            v.copy_(v0)
        vi = v if in_place else (dev(v0, v_dtype) if start else None)
        _lib.check("dw", snnf_lib.snnf_dwconv3x3_lif(
            _lib.step_pointers(xs), _lib.step_pointers(rp) if residual else None, T, N, C, H, W, 1, _lib.dtype_code(dtype), dw.data_ptr(), db.data_ptr(),
            _lib.dtype_code(dtype), _lib.ptr(vi), _lib.dtype_code(v_dtype), sp.data_ptr(), int(sp.stride(0)), v.data_ptr(), *lif, _lib.current_stream(sp.device)))
        assert float(room[0]) == 7.0 and bool((room[1 + T * n:] == 7.0).all())
        got[in_place] = (sp.float().cpu(), v.float().cpu())
        assert torch.equal(got[in_place][0], ref[0])
        if lif is LIF:         # (tau 3 divides)
            assert torch.equal(got[in_place][1], q(ref[1], v_dtype))
    if start:
        assert torch.equal(got[True][1], got[False][1])


@pytest.mark.parametrize("C,H,W,T", [
    (200, 40, 18, 4),        # strips of two workgroups share a row's outputs
    (120, 60, 17, 2),
    (300, 60, 31, 3),
])
@pytest.mark.parametrize("over", ["spikes", "membrane"])
def test_outputs_over_what_is_read(hip_ops, snnf_lib, C, H, W, T, over):
    """Spikes that are written over the residuals, and a final membrane over the last residual: every output is added to once."""
    from triton_snn_fusion_amd import _lib
    g = gen(5290 + C)
    w, b = torch.randint(-64, 65, (C, 1, 3, 3), generator=g) / 64.0, torch.randint(-16, 17, (C,), generator=g) / 64.0
    x = torch.randint(-8, 9, (T, 1, C, H, W), generator=g) / 4.0
    rs = torch.randint(0, 2, (T, 1, C, H, W), generator=g) * 0.75
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), C, *LIF, residuals=list(rs))
    dx, dr, dw, db, code = dev(x, BF16), dev(rs, BF16), dev(w, BF16), dev(b, BF16), _lib.dtype_code(BF16)
    sp = dr if over == "spikes" else torch.empty_like(dx)
    v = dr[T - 1] if over == "membrane" else torch.empty(1, C, H, W, dtype=BF16, device=DEV)
    _lib.check("dw", snnf_lib.snnf_dwconv3x3_lif(
        _lib.step_pointers(list(dx)), _lib.step_pointers(list(dr)), T, 1, C, H, W, 1, code, dw.data_ptr(), db.data_ptr(), code, None, code, sp.data_ptr(), int(sp.stride(0)),
        v.data_ptr(), *LIF, _lib.current_stream(sp.device)))
    assert torch.equal(sp.float().cpu(), ref[0]) and torch.equal(v.float().cpu(), q(ref[1], BF16))
    assert 0.0 < float(ref[0].mean()) < 1.0


@pytest.mark.parametrize("N,C,H,W,T", [
    (4, 125, 20, 11, 5),     # 20000 strips, the fewest of five steps that leave LDS
    (2, 256, 64, 13, 8),     # 65536 strips: one workgroup to each compute unit
    (1, 773, 53, 13, 6),     # more, and fewer than one and a half
    (1, 771, 51, 23, 8),     # between one and a half and two
    (1, 512, 33, 41, 7),     # long rows
])
def test_many_strips_of_odd_rows(hip_ops, snnf_lib, N, C, H, W, T):
    from triton_snn_fusion_amd import _lib
    g = gen(5300 + C + W + T)
    w, b = torch.randint(-64, 65, (C, 1, 3, 3), generator=g) / 64.0, torch.randint(-16, 17, (C,), generator=g) / 64.0
    x = torch.randint(-8, 9, (T, N, C, H, W), generator=g) / 4.0
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), C, *LIF)
    xs, dw, db = dev(x, F16), dev(w, F16), dev(b, F16)
    sp, v = torch.empty((T, N, C, H, W), dtype=F16, device=DEV), torch.empty((N, C, H, W), device=DEV)
    _lib.check("dw", snnf_lib.snnf_dwconv3x3_lif(
        _lib.step_pointers(list(xs)), None, T, N, C, H, W, 1, _lib.dtype_code(F16), dw.data_ptr(), db.data_ptr(), _lib.dtype_code(F16), None, _lib.dtype_code(F32),
        sp.data_ptr(), int(sp.stride(0)), v.data_ptr(), *LIF, _lib.current_stream(sp.device)))
    assert torch.equal(sp.float().cpu(), torch.as_tensor(ref[0])) and torch.equal(v.cpu(), ref[1])
