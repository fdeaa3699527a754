"""Scan and classifier tail where the usual neuron and the others part, and where passes, steps in flight and workgroup sizes end, against the oracle."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import DEV, LIF, gen, q
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
NEURONS = [LIF, (1.0, 0.25, 4.0), (0.75, -1.0, 2.0), (1.0, 0.0, 1.0), (1.0, 0.0, 3.0)]   # usual, usual with a reset potential, soft reset, no leak, a division


@pytest.mark.parametrize("neuron", NEURONS)
@pytest.mark.parametrize("T,n,dtype,vdtype", [(1, 8, BF16, F32), (2, 2056, F16, F16), (3, 13, BF16, F32), (3, 1 << 20, F32, F32), (5, 1032, F32, F32), (8, 4096, BF16, BF16),
                                              (9, 2048, F16, F32), (11, (1 << 20) + 4, F32, F32), (16, 264, BF16, F32), (17, 72, F32, F32)])
def test_scan(snnf_lib, T, n, dtype, vdtype, neuron):
    from triton_snn_fusion_amd import _lib
    g = gen(T * 7 + n)
    x, v0 = q(torch.randn(T, n, generator=g) * 1.5, dtype), q(torch.rand(n, generator=g) * 0.7, vdtype)
    ref, v_ref = [], v0
    for t in range(T):
        fired, v_ref, _ = O.lif_step(x[t], v_ref, *neuron)
        ref.append(fired)
    dx, dv = x.to(DEV, dtype), v0.to(DEV, vdtype)
    s, v = torch.full((T, n), 7.0, device=DEV, dtype=dtype), torch.full((n,), 7.0, device=DEV, dtype=vdtype)
    _lib.check("scan", snnf_lib.snnf_lif_scan(_lib.packed_step_pointers(dx), T, n, _lib.dtype_code(dtype), dv.data_ptr(), _lib.dtype_code(vdtype), s.data_ptr(), n, v.data_ptr(),
                                              *neuron, _lib.current_stream(s.device)))
    # The oracle rounds the product and the sum of a division's step apart, the kernel may not: spikes within 1e-5 of the threshold may differ by a last bit.
    differ = (s.float().cpu() != torch.stack(ref)).float().mean().item()
    assert differ <= (1e-4 if T * n > 1e5 else 0.0), differ
    if vdtype == F32 and differ == 0.0:
        assert torch.allclose(v.cpu(), v_ref, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("neuron", NEURONS)
@pytest.mark.parametrize("T,N,C,HW,K,launches", [
    (4, 3, 2048, 1, 17, 1), (1, 2, 8, 1, 1, 1),              # one pass of 256 threads, full and of a single lane
    (4, 2, 2048 // 8 + 8, 8, 33, 1), (5, 2, 512, 8, 40, 1),  # 512 threads: a little more, and full; eight steps in flight
    (2, 2, 520, 8, 70, 1), (4, 1, 1024, 8, 65, 1),           # 1024 threads
    (1, 2, 1032, 8, 10, 2), (8, 2, 520, 8, 10, 2),           # more neurons, more steps: two launches
    (4, 170, 64, 4, 144, 1), (4, 170, 64, 4, 145, 2),         # three rounds of classes in a workgroup, and four
    (9, 2, 40, 9, 37, 1),                                    # a pass and a step after eight
])
@pytest.mark.parametrize("dtype", [BF16, F32])
def test_tail(snnf_lib, T, N, C, HW, K, launches, dtype, neuron):
    from triton_snn_fusion_amd import _lib
    assert snnf_lib.snnf_lif_pool_linear_launches(T, N, C, HW, 1, K) == launches
    g = gen(T + N * 3 + C + HW)
    x = q(torch.randint(-24, 40, (T, N, C, HW, 1), generator=g) / 16, dtype)
    w, b = q(torch.randint(-8, 9, (K, C), generator=g) / 64, dtype), q(torch.randint(-4, 5, (K,), generator=g) / 4, dtype)
    v0 = torch.randint(0, 12, (N, C, HW, 1), generator=g) / 16
    ref_out, ref_v, _, _ = O.temporal_lif_avgpool_linear(x, v0, w, b, *neuron)
    out, v = torch.full((N, K), 7.0, device=DEV, dtype=dtype), torch.full((N, C, HW, 1), 7.0, device=DEV)
    dx, dw, db, dv = x.to(DEV, dtype), w.to(DEV, dtype), b.to(DEV, dtype), v0.to(DEV)
    space = torch.empty(N * C * 4, dtype=torch.uint8, device=DEV)
    code = _lib.dtype_code(dtype)
    _lib.check("tail", snnf_lib.snnf_lif_pool_linear(
        _lib.packed_step_pointers(dx), T, N, C, HW, 1, code, dv.data_ptr(), _lib.dtype_code(F32), dw.data_ptr(), db.data_ptr(), K, code, out.data_ptr(), v.data_ptr(),
        space.data_ptr(), space.numel(), *neuron, _lib.current_stream(out.device)))
    assert torch.allclose(v.cpu(), ref_v, rtol=1e-5, atol=1e-5)
    tol = 1e-4 if dtype == F32 else 8e-3                     # float32 sums in another order; the outputs' rounding
    assert torch.allclose(out.float().cpu(), ref_out, rtol=tol, atol=tol)
