"""Linear + LIF on rows that start and end anywhere, short rows, and fp32 rows whose terms share a slab, against the oracle."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import DEV, LIF, gen
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("T", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("M,Fin,Fout,pad", [
    (1, 1, 1, 0), (3, 7, 5, 0), (5, 8, 17, 1),       # rows without an octet, of one; row stride beyond the row
    (33, 9, 16, 0), (17, 127, 33, 0), (40, 129, 31, 0), (9, 255, 64, 0), (16, 513, 48, 3),
    (8, 1023, 32, 0), (70, 1025, 20, 0), (200, 264, 96, 4),
    (2, 2055, 16, 0), (130, 1032, 64, 0), (12, 4099, 40, 0),
])
@pytest.mark.parametrize("dtype,shift", [(BF16, 0), (BF16, 1), (F16, 3), (F32, 1)])
def test_rows_of_any_length(snnf_lib, T, M, Fin, Fout, pad, dtype, shift):
    """Operands whose sums are exact in any order; the first row `shift` elements behind a 16-byte address. What lies around the rows is NaN."""
    from triton_snn_fusion_amd import _lib
    g = gen(T + M * 31 + Fin)
    x = torch.randint(-2, 3, (T, M, Fin), generator=g).float()
    w = torch.randint(-8, 9, (Fout, Fin), generator=g) / 8
    b = torch.randint(-4, 5, (Fout,), generator=g) / 4
    left_out = 0.0
    if dtype == F32:                                                       # two bf16 terms each: the product of the low ones is left out (rows of an octet or more)
        x = torch.where(torch.rand(x.shape, generator=g) < 0.5, x.sign(), x) + (x == 0) + torch.randint(0, 2, x.shape, generator=g) / 1024
        w = torch.randint(4, 9, w.shape, generator=g) / 8 * torch.where(w < 0, -1.0, 1.0) + torch.randint(0, 2, w.shape, generator=g) / 1024
        low = [t - t.to(BF16).float() for t in (x, w)]
        left_out = low[0].double() @ low[1].double().T if Fin >= 8 else 0.0
    currents = (x.double() @ w.double().T - left_out + b.double()).float()
    ref, v_ref = [], torch.tensor(0.0)
    for t in range(T):
        fired, v_ref, _ = O.lif_step(currents[t], v_ref, *LIF)
        ref.append(fired)
    room = torch.full((T, M * (Fin + pad) + shift + 16), float("nan"), device=DEV, dtype=dtype)
    rows = room[:, shift:shift + M * (Fin + pad)].view(T, M, Fin + pad)
    rows[..., :Fin] = x.to(DEV, dtype)
    weight = torch.full((Fout * Fin + shift + 16,), float("nan"), device=DEV, dtype=dtype)
    weight[shift:shift + Fout * Fin] = w.to(DEV, dtype).flatten()
    dw, db = weight[shift:], b.to(DEV, dtype)
    s, v = torch.full((T, M, Fout), 7.0, device=DEV, dtype=dtype), torch.full((M, Fout), 7.0, device=DEV)
    _lib.check("linear", snnf_lib.snnf_linear_lif(
        _lib.step_pointers([rows[t] for t in range(T)]), T, M, Fin, Fin + pad, _lib.dtype_code(dtype), dw.data_ptr(), db.data_ptr(), Fout, _lib.dtype_code(dtype), None, 0,
        s.data_ptr(), M * Fout, v.data_ptr(), *LIF, _lib.current_stream(s.device)))
    assert torch.equal(s.float().cpu(), torch.stack(ref))
    assert torch.allclose(v.cpu(), v_ref, rtol=1e-6, atol=1e-6)            # (a neuron that keeps charging ends with more bits than float32 has)


@pytest.mark.parametrize("T,M,Fin,Fout", [
    (1, 80, 1040, 704), (1, 69, 1424, 1361), (1, 80, 2048, 704), (1, 300, 1088, 1200),       # straight from memory, and staged from 2048 on
    (2, 3, 1048, 2505), (2, 65, 1080, 500), (2, 20, 3776, 188), (2, 5, 5456, 10),
])
def test_one_and_two_steps_on_either_side_of_the_line(snnf_lib, T, M, Fin, Fout):
    """K just above multiples of 1024 and of 512, which the two kernels for one and two timesteps of aligned rows go over in rounds and in passes."""
    test_rows_of_any_length(snnf_lib, T, M, Fin, Fout, 0, BF16, 0)


@pytest.mark.parametrize("T,M,Fin,Fout,dtype", [
    (4, 40, 616, 256, BF16), (4, 20, 640, 64, F32),       # three slabs of 256 in a ring of four
    (4, 200, 368, 650, F16), (8, 100, 240, 256, BF16),    # of 128; one in a ring of two
])
def test_one_slab_short_of_the_ring(snnf_lib, T, M, Fin, Fout, dtype):
    """(Whole rows: 16-bit tensors walk the ring all the same, fp32 tensors the slabs that are there.)"""
    test_rows_of_any_length(snnf_lib, T, M, Fin, Fout, 0, dtype, 0)


@pytest.mark.parametrize("dtype,Fin", [(BF16, 25085), (F16, 4001)])
def test_rows_of_eight_timesteps_round_like_those_of_four(snnf_lib, dtype, Fin):
    """Both add K in eight chains, so that the root mean square of what a membrane is off by, which eight timesteps halve and add to like four, is about the same (with half as many chains 1.3 to
    1.45 times as large). 16 rows x 192 features: two such values of equal chains lie within a twentieth or so of each other."""
    from triton_snn_fusion_amd import _lib
    M, Fout, code, off = 16, 192, _lib.dtype_code(dtype), {}
    g = torch.Generator(device=DEV)
    g.manual_seed(5360)
    w = (torch.randn(Fout, Fin, generator=g, device=DEV) / Fin ** 0.5).to(dtype)
    for T in (4, 8):
        x = torch.randn(T, M, Fin, generator=g, device=DEV).to(dtype)
        s, v = torch.empty(T, M, Fout, device=DEV, dtype=dtype), torch.empty(M, Fout, device=DEV)
        _lib.check("linear", snnf_lib.snnf_linear_lif(
            _lib.step_pointers(list(x)), T, M, Fin, Fin, code, w.data_ptr(), None, Fout, code, None, _lib.dtype_code(torch.float32), s.data_ptr(), M * Fout, v.data_ptr(), 1e30, 0.0, 2.0,
            _lib.current_stream(s.device)))
        exact = torch.zeros(M, Fout, dtype=torch.float64, device=DEV)
        for t in range(T):
            exact += (x[t].double() @ w.double().t().contiguous() - exact) / 2
        off[T] = float((v.double() - exact).pow(2).mean().sqrt())
    assert 0.0 < off[8] < 1.15 * off[4], off
