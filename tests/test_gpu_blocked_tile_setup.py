"""How a tile of the blocked convolution starts, at the sizes where that can go wrong: stages smaller than the bias that passes through their LDS, a last
weight fragment that is missing, biases that one of several waves adds, every spike byte, divisors of one. Against the CPU oracle."""
import pytest
import torch

from helpers import LIF, check, dev, gen, q, spikes
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,N,T,dtype,layout", [
    (16, 64, 1, 1, 1, 1, 1, 1, BF16, "bits"),       # a stage of two items, one pixel, one patch
    (8, 8, 1, 2, 1, 1, 1, 1, F16, "bits"),          # a single channel group: pairs of taps
    (16, 40, 1, 1, 1, 1, 40, 2, BF16, "c8"),        # 32 single-pixel planes in a patch
    (64, 96, 7, 7, 3, 1, 3, 4, BF16, "bits"),       # three weight fragments
    (512, 160, 3, 3, 3, 1, 2, 4, F16, "bits"),      # five, K on eight waves
    (128, 128, 28, 28, 3, 1, 16, 4, BF16, "bits"),  # tiles of 64 channels on two waves
    (256, 256, 4, 4, 3, 2, 30, 4, BF16, "bits"),
    (64, 64, 23, 1, 3, 1, 4, 4, F16, "bits"),       # one column
    (64, 64, 1, 23, 3, 1, 4, 3, BF16, "c8"),        # one row
    (64, 64, 40, 40, 3, 1, 60, 4, BF16, "bits"),    # several tiles per wave
])
def test_tiles_start_from_their_bias(snnf_lib, Cin, Cout, H, W, k, s, N, T, dtype, layout):
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    g = gen(8100 + Cin + Cout + H)
    x = torch.stack([spikes((N, Cin, H, W), 0.25, g) for _ in range(T)])
    w, b = q(torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5, dtype), q(torch.randn(Cout, generator=g) * 0.7, dtype)
    p = k // 2
    ref = O.temporal_conv_lif(list(x), w, b, torch.tensor(0.0), (s, s), (p, p), (1, 1), 1, *LIF)
    out, v = B.conv_lif_blocked(B.from_dense(dev(x, dtype), B.BITS if layout == "bits" else B.C8), dev(w, dtype), dev(b, dtype), [s, s], [p, p], LIF,
                                out_layout=B.BITS, want_v=True)
    check(B.to_dense(out), v, ref, what=f"{Cin}->{Cout} {H}x{W} T={T}")


@pytest.mark.parametrize("dtype", [BF16, F16])
def test_every_spike_byte(snnf_lib, dtype):
    """256 pixels with all patterns of eight channels, through the identity: the sums are the spikes themselves."""
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    bits = (torch.arange(256)[None, :] >> torch.arange(8)[:, None]) & 1                     # [8, 256]
    x = torch.cat([bits, bits.flip(1)]).reshape(1, 1, 16, 16, 16).float()
    eye = torch.eye(16).reshape(16, 16, 1, 1)
    out, _ = B.conv_lif_blocked(B.from_dense(dev(x, dtype), B.BITS), dev(eye, dtype), dev(torch.zeros(16), dtype), [1, 1], [0, 0], None, out_layout=B.NCHW)
    assert torch.equal(B.to_dense(out).float().cpu(), x)
