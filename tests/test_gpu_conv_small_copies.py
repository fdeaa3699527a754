"""The line of the dense rule for layers whose copy is small: either side of it, and the moved layer against the matrix kernel and the oracle."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import DEV, LIF, dev, gen, spikes
from oracle import snn_oracle as O

BF16 = torch.bfloat16


@pytest.mark.parametrize("T,N,Cin,Cout,H,moves", [(4, 16, 128, 128, 28, True), (4, 32, 128, 128, 28, False), (1, 26, 128, 128, 28, True), (1, 27, 128, 128, 28, False),
                                                  (4, 8, 64, 64, 32, True), (4, 16, 64, 64, 56, False)])
def test_line(snnf_lib, T, N, Cin, Cout, H, moves):
    assert (snnf_lib.snnf_conv_lif_scratch_bytes(T, N, Cin, H, H, 1, Cout, 3, 3, 1, 1, 1, 1, 0, 0) > 0) == moves


@pytest.mark.gpu
@pytest.mark.parametrize("residual", [False, True])
def test_moved_layer(hip_ops, residual):
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    S = torch.ops.snn_custom
    g = gen(12)
    T, N, C, H = 4, 3, 128, 28
    x = [spikes((N, C, H, H), 0.2, g) for _ in range(T)]
    r = [spikes((N, C, H, H), 0.2, g) for _ in range(T)] if residual else None
    w = (torch.randn(C, C, 3, 3, generator=g) * 16).round() / 128          # (exact sums: bit for bit the oracle)
    b = (torch.randn(C, generator=g) * 2).round() / 16
    ref = O.temporal_conv_lif(x, w, b, torch.tensor(0.0), (1, 1), (1, 1), (1, 1), 1, *LIF, residuals=r)
    args = (dev(w, BF16), dev(b, BF16), torch.zeros((), device=DEV), [1, 1], [1, 1], [1, 1], 1, *LIF, False)
    dx = [dev(t, BF16) for t in x]
    s, v = S.fused_temporal_conv_lif_state(dx, *args) if r is None else S.fused_temporal_conv_add_lif_state(dx, [dev(t, BF16) for t in r], *args)
    assert CB.last_conv_plan()["ran"] == "blocked", CB.last_conv_plan()
    assert torch.equal(s.float().cpu(), ref[0]) and torch.allclose(v.cpu(), ref[1], rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("T,N,Cin,Cout,H,W,residual,moves", [
    (4, 16, 128, 128, 28, 28, 1, True),        # 1792 waves of 2048
    (4, 11, 64, 64, 56, 56, 1, False),         # 1078
    (2, 58, 32, 512, 32, 32, 1, False),        # more than two rounds
    (4, 20, 64, 64, 48, 28, 0, False),         # patches of four columns
    (4, 16, 128, 64, 28, 28, 1, False),        # few output channels for the copy
    (1, 8, 64, 128, 80, 28, 1, True),          # one timestep
    (4, 8, 64, 64, 32, 32, 0, True),           # narrow tiles
])
def test_layers_that_fill_the_waves(snnf_lib, T, N, Cin, Cout, H, W, residual, moves):
    """Beyond the usual line only layers move whose plan on the blocked kernel is a good one."""
    assert (snnf_lib.snnf_conv_lif_scratch_bytes(T, N, Cin, H, W, 1, Cout, 3, 3, 1, 1, 1, 1, 0, residual) > 0) == moves
