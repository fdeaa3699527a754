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
