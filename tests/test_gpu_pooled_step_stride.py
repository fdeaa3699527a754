"""Pooled spikes whose timesteps do not lie side by side: any step stride that the entry point takes, by every kernel behind it, against the contiguous call."""
import pytest
import torch

import triton_snn_fusion_amd  # noqa: F401
from helpers import DEV, LIF, dev, gen, spikes

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
T = 4
GIB = 1 << 30


@pytest.mark.parametrize("Cin,Cout,H,N,layout,few", [
    (64, 64, 32, 24, "bits", False),         # a wave per tile
    (128, 128, 16, 8, "bits", False),        # a tile's sums shared by several waves
    (3, 64, 32, 2, "frame", False),          # a dense frame for all timesteps
    (256, 256, 8, 1, "bits", True),          # few pixels
])
@pytest.mark.parametrize("stride", ["gap", 3 * GIB // 2, -(3 * GIB // 2), "back"])
def test_steps_anywhere(hip_ops, Cin, Cout, H, N, layout, few, stride):
    from triton_snn_fusion_amd import _lib
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    g = gen(Cin + H)
    w = dev((torch.randn(Cout, Cin, 3, 3, generator=g) * 16).round() / 64, BF16)
    b = dev((torch.randn(Cout, generator=g) * 2).round() / 16, BF16)
    if layout == "frame":
        x = B.from_dense(dev(torch.randint(-32, 33, (N, Cin, H, H), generator=g) / 16.0, BF16), B.C8, shared=True)
        x.T = T
    else:
        x = B.from_dense(dev(spikes((T, N, Cin, H, H), 0.2, g), BF16), B.BITS)
    want, _ = B.conv_lif_blocked_avgpool(x, w, b, [1, 1], [1, 1], LIF)
    assert ("few" in B.last_conv_plan()) == few, B.last_conv_plan()
    want = want.data.contiguous().view(torch.uint8).reshape(T, -1)
    frame = want.shape[1]
    assert 0.0 < float((want != 0).float().mean())
    step = {"gap": frame + 24, "back": -(frame + 8)}.get(stride, stride)
    store = torch.empty(3 * abs(step) + frame, dtype=torch.uint8, device=DEV)
    starts = [(t if step > 0 else 3 - t) * abs(step) for t in range(T)]
    for at in starts:
        store[at:at + frame].fill_(0x55)
    if abs(step) < GIB:
        store.fill_(0x55)
    packed = B._packed_weight(w, b, BF16)
    _lib.check("snnf_conv_lif_blocked_avgpool", _lib.lib().snnf_conv_lif_blocked_avgpool(
        x.step_pointers(), x.layout, T, N, Cin, H, H, _lib.dtype_code(BF16), packed.data_ptr(), Cout, 3, 3, 1, 1, 1, 1,
        store.data_ptr() + starts[0], step, None, *LIF, _lib.current_stream(store.device)))
    for t, at in enumerate(starts):
        assert torch.equal(store[at:at + frame], want[t]), t
    if abs(step) < GIB:                                                    # nothing between the steps is written
        for at in sorted(starts)[:3]:
            assert bool((store[at + frame:at + abs(step)] == 0x55).all())
