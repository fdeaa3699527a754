"""The final membrane in the memory of the initial one (`v_out` == `v_init`, which the C ABI allows): spikes and membrane are those of a
call with memory of its own, bit for bit."""
import pytest
import torch

from helpers import DEV, LIF, gen, spikes

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def both_ways(call, v0):
    """call(v_init, v_out) -> outputs, with and without memory shared between the two."""
    v_init, v_out = v0.clone(), torch.full_like(v0, float("nan"))
    want = call(v_init, v_out)
    assert torch.equal(v_init, v0) and not torch.equal(v_out, v0)
    v = v0.clone()
    got = call(v, v)
    assert torch.equal(v, v_out) and torch.equal(got, want) and bool(want.any())


@pytest.mark.parametrize("N,C,HW,K,dtype,v_dtype,launches", [
    (2, 64, 7, 1000, BF16, F32, 1),     # one launch with separate memory: 63 class ranges read a sample's membrane
    (300, 512, 2, 40, F32, F32, 1),     # one class range per sample
    (3, 1024, 7, 33, F16, F16, 2),
])
@pytest.mark.parametrize("static", [False, True])
def test_tail(snnf_lib, N, C, HW, K, dtype, v_dtype, launches, static):
    from triton_snn_fusion_amd import _lib
    assert snnf_lib.snnf_lif_pool_linear_launches(4, N, C, HW, HW, K) == launches
    g = gen(9000 + N)
    xs = [(torch.randn(N, C, HW, HW, generator=g) + 0.5).to(DEV, dtype) for _ in range(4)]
    w, b = torch.randn(K, C, generator=g).to(DEV, dtype), torch.randn(K, generator=g).to(DEV, dtype)
    space = torch.empty(N * C * 4, dtype=torch.uint8, device=DEV)

    def call(v_init, v_out):
        out = torch.empty(N, K, device=DEV, dtype=dtype)
        code = _lib.dtype_code(dtype)
        args = [_lib.step_pointers(xs), 4, N, C, HW, HW, code, v_init.data_ptr(), _lib.dtype_code(v_dtype), w.data_ptr(), b.data_ptr(), K, code,
                out.data_ptr(), v_out.data_ptr()]
        if static: _lib.check("tail", snnf_lib.snnf_lif_pool_linear_static(*args, *LIF, _lib.current_stream(out.device)))
        else: _lib.check("tail", snnf_lib.snnf_lif_pool_linear(*args, space.data_ptr(), space.numel(), *LIF, _lib.current_stream(out.device)))
        return out

    both_ways(call, (torch.rand(N, C, HW, HW, generator=g) * 0.9).to(DEV, v_dtype))


@pytest.mark.parametrize("Cin,Cout,H,W,k,T,N,dtype,v_dtype,residual,kernel,blocked", [
    (64, 64, 16, 16, 3, 4, 2, BF16, F32, True, "matrix", False),         # whole tiles
    (64, 64, 16, 16, 3, 6, 2, BF16, F32, False, "matrix", False),        # ... a window per launch
    (72, 40, 9, 7, 3, 4, 2, F16, F32, True, "matrix", False),            # masked tiles
    (64, 128, 8, 8, 1, 4, 3, BF16, F32, False, "pointwise", False),
    (64, 72, 7, 9, 1, 5, 2, BF16, F32, True, "pointwise", False),
    (20, 24, 9, 9, 3, 3, 2, BF16, BF16, False, None, False),             # a partly filled channel group
    (12, 33, 6, 7, 3, 4, 2, F32, F32, True, None, False),
    (72, 40, 9, 7, 3, 4, 2, BF16, F32, True, None, True),
    (72, 104, 9, 7, 3, 7, 2, F16, F32, True, None, True),                # two windows, the membrane between them in v_out
    (72, 104, 9, 7, 3, 7, 2, F16, F16, False, None, True),               # ... in scratch memory
    (40, 34, 33, 31, 3, 9, 8, F32, F32, True, None, True),
])
def test_convolution(snnf_lib, Cin, Cout, H, W, k, T, N, dtype, v_dtype, residual, kernel, blocked):
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    g, p, code, v_code = gen(9100 + Cin + T), k // 2, _lib.dtype_code(dtype), _lib.dtype_code(v_dtype)
    xs = [spikes((N, Cin, H, W), 0.25, g).to(DEV, dtype) for _ in range(T)]
    rs = [spikes((N, Cout, H, W), 0.25, g).to(DEV, dtype) for _ in range(T)] if residual else None
    w, b = (torch.randn(Cout, Cin, k, k, generator=g) * 3.0 * (2.0 / (Cin * k * k)) ** 0.5).to(DEV, dtype), torch.zeros(Cout, device=DEV, dtype=dtype)
    packed = CB._packed_weight(w, b, dtype)
    need = snnf_lib.snnf_conv_lif_scratch_bytes(T, N, Cin, H, W, code, Cout, k, k, 1, 1, p, p, v_code, int(residual)) if blocked else 0
    space = torch.empty(need, dtype=torch.uint8, device=DEV)

    def call(v_init, v_out):
        out = torch.empty(T, N, Cout, H, W, device=DEV, dtype=dtype)
        _lib.check("conv", snnf_lib.snnf_conv_lif_ws(
            _lib.step_pointers(xs), _lib.step_pointers(rs) if residual else None, T, N, Cin, H, W, code, packed.data_ptr(), Cout, k, k, 1, 1, p, p,
            v_init.data_ptr(), v_code, out.data_ptr(), int(out.stride(0)), v_out.data_ptr(), *LIF, space.data_ptr() if need else None, need,
            _lib.current_stream(out.device)))
        plan = CB.last_conv_plan()
        assert (plan.get("ran") == "blocked") == blocked and kernel in (None, plan["kernel"]), plan
        return out

    both_ways(call, (torch.rand(N, Cout, H, W, generator=g) * 0.9).to(DEV, v_dtype))


@pytest.mark.parametrize("T,Cin,Cout,H,W,N,bits_out", [(4, 64, 64, 12, 12, 2, True), (7, 128, 40, 9, 7, 3, True), (6, 64, 72, 16, 16, 8, False)])
def test_convolution_on_internal_layouts(snnf_lib, T, Cin, Cout, H, W, N, bits_out):
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B, hip_convlif_backend as CB
    g = gen(9200 + T)
    x = B.from_dense(torch.stack([spikes((N, Cin, H, W), 0.25, g) for _ in range(T)]).to(DEV, BF16), B.BITS)
    w = (torch.randn(Cout, Cin, 3, 3, generator=g) * 3.0 * (2.0 / (Cin * 9)) ** 0.5).to(DEV, BF16)
    packed, step = CB._packed_weight(w, torch.zeros(Cout, device=DEV, dtype=BF16), BF16), N * (Cin // 8) * H * W
    layout = B.BITS if bits_out else B.NCHW
    steps = [x.data[t] for t in range(T)]
    assert steps[0].numel() * steps[0].element_size() == step

    def call(v_init, v_out):
        out = torch.zeros((T, N, Cout // 8, H, W) if bits_out else (T, N, Cout, H, W), device=DEV, dtype=torch.uint8 if bits_out else BF16)
        _lib.check("blocked", snnf_lib.snnf_conv_lif_blocked(
            _lib.step_pointers(steps), B.BITS, None, 0, T, N, Cin, H, W, _lib.dtype_code(BF16), packed.data_ptr(), Cout, 3, 3, 1, 1, 1, 1, v_init.data_ptr(),
            out.data_ptr(), layout, out.stride(0) * out.element_size(), v_out.data_ptr(), 1, *LIF, _lib.current_stream(out.device)))
        return out

    both_ways(call, (torch.rand(N, Cout, H, W, generator=g) * 0.9).to(DEV))


@pytest.mark.parametrize("op,shape,T,dtype,v_dtype", [
    ("scan", (3, 40, 9, 7), 5, BF16, BF16), ("scan", (2, 64, 8, 8), 20, F32, F32),               # 20 steps: two launches
    ("depthwise", (3, 24, 14, 14), 4, BF16, F32), ("depthwise", (2, 40, 9, 7), 18, F16, F32), ("depthwise", (2, 16, 12, 12), 3, F32, F32),
    ("linear", (9, 100, 33), 4, BF16, F32), ("linear", (64, 2048, 96), 8, BF16, BF16), ("linear", (2, 64, 10), 2, F32, F32),
    ("linear", (16, 4096, 64), 4, F16, F32),                                                     # partial sums in the workspace
])
def test_other_operators(snnf_lib, op, shape, T, dtype, v_dtype):
    from triton_snn_fusion_amd import _lib
    g, code, v_code = gen(9300 + T + shape[1]), _lib.dtype_code(dtype), _lib.dtype_code(v_dtype)
    x_shape, v_shape = (shape[:2], (shape[0], shape[2])) if op == "linear" else (shape, shape)
    xs = [(spikes(x_shape, 0.25, g) * (4.0 if op == "scan" else 1.0)).to(DEV, dtype) for _ in range(T)]
    w = {"scan": None, "depthwise": torch.randn(shape[1], 1, 3, 3, generator=g), "linear": torch.randn(shape[-1], shape[1], generator=g) * 4.0 * shape[1] ** -0.5}[op]
    w = None if w is None else w.to(DEV, dtype)
    b = None if w is None else torch.zeros(w.shape[0], device=DEV, dtype=dtype)
    need = int(snnf_lib.snnf_linear_lif_workspace_bytes(T, *shape)) if op == "linear" else 0
    space = torch.zeros(max(need, 16), dtype=torch.uint8, device=DEV)

    def call(v_init, v_out):
        out = torch.empty(T, *v_shape, device=DEV, dtype=dtype)
        steps, stream = _lib.step_pointers(xs), _lib.current_stream(out.device)
        tail = (v_init.data_ptr(), v_code, out.data_ptr(), int(out.stride(0)), v_out.data_ptr(), *LIF)
        if op == "scan": rc = snnf_lib.snnf_lif_scan(steps, T, v_out.numel(), code, *tail, stream)
        elif op == "depthwise": rc = snnf_lib.snnf_dwconv3x3_lif(steps, None, T, *shape, 1, code, w.data_ptr(), b.data_ptr(), code, *tail, stream)
        else: rc = snnf_lib.snnf_linear_lif_ws(steps, T, shape[0], shape[1], shape[1], code, w.data_ptr(), b.data_ptr(), shape[2], code, *tail,
                                               space.data_ptr() if need else None, need, stream)
        _lib.check(op, rc)
        return out

    both_ways(call, (torch.rand(v_shape, generator=g) * 0.9).to(DEV, v_dtype))
