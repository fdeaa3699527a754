"""Convolutions of fp32 tensors on the blocked kernel (two bf16 terms per value): against the CPU oracle, against float64 and against the
dense kernels, where low terms are absent, everywhere or in a single pixel, at the edges of channel groups, tiles, windows and epilogues."""
import pytest
import torch

from helpers import DEV, LIF, check, dev, gen, spikes
from oracle import snn_oracle as O

pytestmark = pytest.mark.gpu
F32 = torch.float32
SOFT, SLOW, RESET = (1.0, -1.0, 2.0), (0.8, 0.0, 4.0), (1.0, 0.25, 2.0)

CASES = [  # (Cin, Cout, H, W, k, stride, T, N, residual, tensor v_init, low terms in, neuron)
    (64, 64, 32, 32, 3, 1, 4, 2, False, False, "none", LIF),       # K shared by waves
    (64, 64, 56, 56, 3, 1, 4, 7, True, False, "one", LIF),         # a tile per wave; one pixel with a low term
    (64, 64, 24, 24, 3, 1, 4, 3, True, True, "all", LIF),
    (41, 72, 8, 14, 3, 1, 4, 5, True, False, "one", LIF),          # a partly filled channel group
    (20, 33, 5, 7, 3, 1, 3, 2, True, True, "all", LIF),            # 33 channels: single channels are masked
    (17, 30, 9, 5, 5, 2, 5, 1, False, True, "all", LIF),           # two windows
    (6, 10, 11, 9, 3, 1, 16, 2, True, False, "all", LIF),          # pairs of taps, four windows
    (12, 40, 6, 6, 7, 2, 2, 3, False, True, "one", LIF),           # two timesteps
    (64, 128, 7, 7, 1, 1, 4, 3, True, False, "all", LIF),          # pointwise
    (99, 130, 1, 1, 1, 1, 1, 9, False, False, "all", LIF),         # one pixel, one timestep
    (512, 64, 2, 2, 3, 1, 4, 9, False, False, "one", LIF),         # several images per tile
    (256, 96, 7, 7, 3, 2, 6, 2, True, True, "none", LIF),
    (40, 24, 10, 10, 3, 1, 5, 2, True, True, "all", SOFT),         # the general epilogue
    (40, 26, 10, 10, 3, 1, 4, 1, True, False, "one", SLOW),
    (64, 64, 32, 32, 3, 1, 2, 8, True, True, "all", SOFT),
    (40, 24, 10, 10, 3, 1, 4, 2, False, True, "none", RESET),
]


def operands(Cin, Cout, H, W, k, s, T, N, residual, tensor_v, low, seed):
    g = gen(seed)
    Ho, Wo = (H + 2 * (k // 2) - k) // s + 1, (W + 2 * (k // 2) - k) // s + 1
    xs = [spikes((N, Cin, H, W), 0.25, g) for _ in range(T)]
    if low == "all":
        xs = [x + 0.3 * torch.randn(x.shape, generator=g) for x in xs]
    elif low == "one":
        xs[-1][N - 1, Cin - 1, H - 1, 0] = 1.0 + 2.0 ** -12        # bf16 holds seven bits behind the point
    w = torch.randn(Cout, Cin, k, k, generator=g) * 2.0 * (2.0 / (Cin * k * k)) ** 0.5
    b = torch.randn(Cout, generator=g) * 0.1
    rs = [torch.randn(N, Cout, Ho, Wo, generator=g) * 0.3 for _ in range(T)] if residual else None
    v0 = torch.randn(N, Cout, Ho, Wo, generator=g) * 0.3 if tensor_v else torch.tensor(0.0)
    return xs, w, b, rs, v0


def run(lib, xs, w, b, rs, v0, k, s, lif, fill, given=None):
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    T, (N, Cin, H, W), Cout, p = len(xs), xs[0].shape, w.shape[0], k // 2
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    need = lib.snnf_conv_lif_scratch_bytes(T, N, Cin, H, W, 0, Cout, k, k, s, s, p, p, 0, int(rs is not None))
    step = N * -(-Cin // 8) * H * W * 16
    assert need == T * (2 * step + -(-step // 4096) * 4)                # both terms, and a byte per 64 items in whole dwords
    given = need if given is None else given
    dx, dr, dv = [dev(x, F32) for x in xs], [dev(r, F32) for r in rs] if rs is not None else None, dev(v0, F32) if v0.dim() else None
    packed = CB._packed_weight(dev(w, F32), dev(b, F32), F32)
    workspace = torch.full((need,), fill, dtype=torch.uint8, device=DEV)
    sp, v = torch.empty(T, N, Cout, Ho, Wo, device=DEV), torch.empty(N, Cout, Ho, Wo, device=DEV)
    _lib.check("ws", lib.snnf_conv_lif_ws(
        _lib.step_pointers(dx), _lib.step_pointers(dr) if dr is not None else None, T, N, Cin, H, W, 0, packed.data_ptr(), Cout, k, k, s, s, p, p,
        _lib.ptr(dv), 0, sp.data_ptr(), int(sp.stride(0)), v.data_ptr(), *lif, workspace.data_ptr(), given, _lib.current_stream(sp.device)))
    assert (CB.last_conv_plan().get("ran") == "blocked") == (given >= need), CB.last_conv_plan()
    return sp, v


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,T,N,residual,tensor_v,low,lif", CASES)
def test_fp32_convolution_on_the_blocked_kernel(snnf_lib, Cin, Cout, H, W, k, s, T, N, residual, tensor_v, low, lif):
    xs, w, b, rs, v0 = operands(Cin, Cout, H, W, k, s, T, N, residual, tensor_v, low, 6000 + Cin + Cout + H + T)
    p = k // 2
    ref = O.temporal_conv_lif(xs, w, b, v0, (s, s), (p, p), (1, 1), 1, *lif, residuals=rs)
    for fill in (255, 0):                                                # scratch of NaN patterns (every flag set), and of zeros
        sp, v = run(snnf_lib, xs, w, b, rs, v0, k, s, lif, fill)
        check(sp, v, ref, v_threshold=lif[0], what=f"fp32 {Cin}->{Cout} {H}x{W} {low}")


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,T,N,residual,tensor_v,low,lif", [c for c in CASES if c[11] == LIF])
def test_no_further_from_float64_than_the_dense_kernels(snnf_lib, Cin, Cout, H, W, k, s, T, N, residual, tensor_v, low, lif):
    """Both routes multiply the same three of the four products of the terms; a silent neuron leaves the sums in its membrane. What may
    differ is the order of the fp32 additions: a random walk of roundings on either side, hence the margin of a quarter."""
    xs, w, b, rs, v0 = operands(Cin, Cout, H, W, k, s, T, N, residual, tensor_v, low, 6100 + Cin + Cout + H + T)
    p, v64 = k // 2, v0.double()
    for t, x in enumerate(xs):
        v64 = (v64 + torch.nn.functional.conv2d(x.double(), w.double(), b.double(), s, p) + (rs[t].double() if residual else 0)) / 2
    error = {}
    for name, given in (("blocked", None), ("dense", 0)):
        sp, v = run(snnf_lib, xs, w, b, rs, v0, k, s, (1e9, 0.0, 2.0), 255, given)
        assert not sp.any()
        error[name] = float((v.double().cpu() - v64).norm() / v64.norm())
    assert error["blocked"] <= 1.25 * error["dense"] + 2.0 ** -24, error


def test_layers_of_fp32_tensors_that_stay(snnf_lib):
    asks = snnf_lib.snnf_conv_lif_scratch_bytes
    assert asks(4, 16, 64, 56, 56, 0, 128, 1, 1, 1, 1, 0, 0, 0, 0) == 0          # pointwise, few products, many outputs
    assert asks(4, 8, 64, 28, 28, 0, 128, 1, 1, 1, 1, 0, 0, 0, 0) > 0
    assert asks(17, 8, 20, 9, 9, 0, 24, 3, 3, 1, 1, 1, 1, 0, 0) == 0             # more timesteps than one launch takes


def test_infinities_and_nan_reach_the_same_neurons(snnf_lib):
    """Not-a-number and infinite inputs: the neurons they reach hold no number on either route, all others are untouched."""
    xs, w, b, rs, v0 = operands(24, 40, 9, 9, 3, 1, 4, 2, False, False, "none", 6200)
    xs[1][0, 3, 4, 4], xs[2][1, 5, 0, 0] = float("nan"), float("inf")
    got = run(snnf_lib, xs, w, b, rs, v0, 3, 1, LIF, 255)
    want = run(snnf_lib, xs, w, b, rs, v0, 3, 1, LIF, 255, 0)
    assert torch.equal(got[1].isnan(), want[1].isnan()) and got[1].isnan().any()
    assert torch.equal(got[0], want[0]) and torch.allclose(got[1], want[1], rtol=1e-5, atol=1e-6, equal_nan=True)


@pytest.mark.parametrize("Cin,Cout,H,W,k,s,T,N,groups", [
    (16, 32, 40, 24, 3, 1, 4, 2, None),         # tiles of part of an image
    (40, 24, 23, 31, 3, 1, 3, 2, (0, 3, 4)),    # flags of 64 items across rows and channel groups; a stage with a single group
    (24, 24, 64, 8, 5, 2, 5, 1, (1, 2)),        # two windows, the last of one timestep
    (600, 16, 9, 14, 1, 1, 2, 2, (0, 10, 63, 64, 73, 74)),    # more than 64 channel groups
    (6, 16, 33, 33, 3, 1, 4, 1, None),          # pairs of taps
    (64, 16, 4, 4, 3, 1, 4, 5, (0, 7)),         # several images per tile
])
def test_a_low_term_counts_wherever_it_is(snnf_lib, Cin, Cout, H, W, k, s, T, N, groups):
    """One input per call, 1 + 2^-9 (terms 1 and 2^-9), between zeros: an output that it reaches is one product, whose dropped part, the
    product of the two low terms, is 2^-16 of it or less. The sums of the silent neuron are scaled by powers of two."""
    g = gen(6300 + Cin)
    Ho, Wo = (H + 2 * (k // 2) - k) // s + 1, (W + 2 * (k // 2) - k) // s + 1
    w = torch.randn(Cout, Cin, k, k, generator=g).sign() * (torch.rand(Cout, Cin, k, k, generator=g) + 0.5)
    places = [(h, x) for h in sorted({0, 1, H // 2, H - 2, H - 1}) for x in (0, W // 2, W - 1)]
    for i, (h, x) in enumerate(places):
        xs = [torch.zeros(N, Cin, H, W) for _ in range(T)]
        group = (groups or range(-(-Cin // 8)))[i % len(groups or range(-(-Cin // 8)))]
        xs[i % T][i % N, min(group * 8 + i % 8, Cin - 1), h, x] = 1.0 + 2.0 ** -9
        got = run(snnf_lib, xs, w, torch.zeros(Cout), None, torch.tensor(0.0), k, s, (1e9, 0.0, 2.0), 255)[1].double().cpu()
        v64 = torch.zeros(N, Cout, Ho, Wo, dtype=torch.float64)
        for step in xs:
            v64 = (v64 + torch.nn.functional.conv2d(step.double(), w.double(), None, s, k // 2)) / 2
        assert torch.all((got - v64).abs() <= v64.abs() * 2.0 ** -15), (h, x, group)
