"""Convolutions whose scratch memory the allocator does not have: they run on the dense kernels, which need none. Weights are fixed-point
numbers whose sums are exact in fp32 in any order, so the results are those of the blocked route bit for bit."""
import contextlib

import pytest
import torch

from helpers import DEV, gen, spikes

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
SAME = ([1, 1], [1, 1], [1, 1], 1)
LIF = (1.0, 0.0, 2.0, False)


@contextlib.contextmanager
def memory_limit(room):
    """The allocator gets `room` bytes beyond what is in use."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + room) / torch.cuda.mem_get_info()[1])
    try:
        yield
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


def operands(T, dtype, tensor_v=None, residual=False):
    g = gen(8100 + T)
    w = torch.randint(-512, 513, (16, 512, 3, 3), generator=g) / 8192
    b = torch.randint(-64, 65, (16,), generator=g) / 1024
    N = 16 if T > 1 else 64                                     # scratch areas of 100 MB and more
    xs = [spikes((N, 512, 40, 40), 0.25, g).to(DEV, dtype) for _ in range(T)]
    rs = [spikes((N, 16, 40, 40), 0.25, g).to(DEV, dtype) for _ in range(T)] if residual else None
    v0 = torch.zeros((), device=DEV) if tensor_v is None else (torch.randint(-512, 513, (N, 16, 40, 40), generator=g) / 1024).to(DEV, tensor_v)
    return xs, rs, w.to(DEV, dtype), b.to(DEV, dtype), v0


@pytest.mark.parametrize("T,dtype,tensor_v,residual", [
    (4, BF16, None, False),
    (4, F32, None, True),           # two C8 tensors
    (6, F16, F16, False),           # a 16-bit membrane over several windows, in float32 between them
    (4, BF16, BF16, True),          # ... over one window of the blocked kernel, and two of the dense one
    (1, BF16, BF16, False),
])
def test_no_scratch_memory_left(hip_ops, T, dtype, tensor_v, residual):
    from triton_snn_fusion_amd import _dispatch
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    S = torch.ops.snn_custom
    xs, rs, w, b, v0 = operands(T, dtype, tensor_v, residual)
    call = lambda: (S.fused_temporal_conv_add_lif_state(xs, rs, w, b, v0, *SAME, *LIF) if residual
                    else S.fused_temporal_conv_lif_state(xs, w, b, v0, *SAME, *LIF))
    want = call()
    assert CB.last_conv_plan().get("ran") == "blocked"
    call()                                                      # the native implementation
    assert CB.last_conv_plan().get("ran") == "blocked" and 0.0 < float(want[0].float().mean()) < 0.9
    for python in (False, True):
        hip_ops.configure_fused_op("hip", strict_triton=True, verbose=python)
        hits = sum(_dispatch.module().hits())
        with memory_limit(24 << 20):                            # room for the outputs
            got = call()
        assert CB.last_conv_plan().get("ran") != "blocked", CB.last_conv_plan()
        assert sum(_dispatch.module().hits()) - hits == (0 if python else 1)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and got[1].dtype == want[1].dtype
    hip_ops.configure_fused_op("hip", strict_triton=True)
    call()
    assert CB.last_conv_plan().get("ran") == "blocked"


def test_no_scratch_memory_left_without_a_neuron(hip_ops):
    from triton_snn_fusion_amd import _dispatch
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    xs, _, w, b, _ = operands(4, BF16)
    x, native = torch.stack(xs), _dispatch.module()
    want = CB.run_hip_conv_bias_frames(x, w, b, [1, 1], [1, 1])
    assert CB.last_conv_plan().get("ran") == "blocked"
    with memory_limit(24 << 20):
        got = native.dense_conv_bias(x, w, b, [1, 1], [1, 1], -1)
    assert got is not None and CB.last_conv_plan().get("ran") != "blocked" and torch.equal(got, want)
    del got
    with memory_limit(24 << 20):
        got = CB.run_hip_temporal_conv_bias(list(x.unbind(0)), w, b, [1, 1], [1, 1])
    assert CB.last_conv_plan().get("ran") != "blocked" and torch.equal(got, want)
