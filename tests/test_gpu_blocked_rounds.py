"""Launches of several rounds of waves: which take every compute unit, and that an image's spikes do not depend on how the tiles are dealt."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import DEV, LIF, gen

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


@pytest.mark.parametrize("kind,N,grid", [
    ("64 at 56", 52, 256),        # 2.49 rounds: every unit
    ("64 at 56", 60, 245),        # 2.87: full rounds on fewer
    ("64 at 56", 36, 221),        # two rounds
    ("stem", 16, 512),            # 1.53 rounds of two workgroups a unit
    ("stem", 20, 490),            # 1.91
])
def test_last_round(snnf_lib, kind, N, grid):
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the shapes sit at the edges of 256 compute units")
    g = gen(N)
    if kind == "stem":
        x = (torch.randint(-128, 128, (N, 3, 224, 224), generator=g).float() / 64).to(DEV, BF16)
        w, s, p = torch.randint(-16, 17, (64, 3, 7, 7), generator=g) / 128, [2, 2], [3, 3]
        operand = lambda t: B.input_frame(t, 4)
    else:
        x = (torch.rand((4, N, 64, 56, 56), generator=g) < 0.2).to(DEV, BF16)
        w, s, p = torch.randint(-16, 17, (64, 64, 3, 3), generator=g) / 128, [1, 1], [1, 1]
        operand = lambda t: B.from_dense(t, B.BITS)
    w, b = w.to(DEV, BF16), torch.zeros(64, device=DEV, dtype=BF16)
    out, _ = B.conv_lif_blocked(operand(x), w, b, s, p, LIF, out_layout=B.BITS)
    assert int(B.last_conv_plan()["grid"]) == grid, B.last_conv_plan()
    got = B.to_dense(out)
    assert 0.01 < float(got.float().mean()) < 0.9
    for n in (0, N // 2, N - 1):       # (sums of whole multiples of 2^-13: exact in any order)
        one = (x[n:n + 1] if kind == "stem" else x[:, n:n + 1]).contiguous()
        alone, _ = B.conv_lif_blocked(operand(one), w, b, s, p, LIF, out_layout=B.BITS)
        assert torch.equal(got[:, n:n + 1], B.to_dense(alone)), n
