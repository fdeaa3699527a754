"""Membranes stored in bfloat16: the conversion instruction against torch's rounding, bit for bit, over all kinds of values."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import DEV, gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exponents", [None, (0, 2), (1, 12), (240, 254), (255, 255)])       # all bit patterns; denormals; small; overflow; infinities and NaN
@pytest.mark.parametrize("n", [8, 4096 + 3, 1 << 18])
def test_sums_rounded_to_bf16(hip_ops, exponents, n):
    g = gen(n)
    bits = [torch.randint(-(1 << 15), 1 << 15, (n,), generator=g).to(torch.int16) for _ in range(2)]
    if exponents is not None:
        lo, hi = exponents
        bits = [(b & torch.tensor(0x807f - (1 << 16), dtype=torch.int16)) | (torch.randint(lo, hi + 1, (n,), generator=g) << 7).to(torch.int16) for b in bits]
    v, x = (b.view(torch.bfloat16) for b in bits)
    h = v.float() + x.float()                                  # exact to 24 bits, then one rounding to 8
    fired = h >= 1e30
    want = torch.where(fired, torch.zeros(()), h).to(torch.bfloat16)
    s, got = torch.ops.snn_custom.lif_forward_state(x.to(DEV), v.to(DEV), 1e30, 0.0, 1.0, False)
    assert got.dtype == torch.bfloat16 and torch.equal(s.cpu(), fired.to(torch.bfloat16))
    got = got.cpu()
    assert torch.equal(got.isnan(), want.isnan())
    real = ~want.isnan()
    assert torch.equal(got.view(torch.int16)[real], want.view(torch.int16)[real])
