"""The native dispatch (csrc/host/snnf_dispatch.cpp): a call of a known signature returns bit for bit what the first call (the
Python implementation) returned, counts the same statistics, follows in-place weight updates and replaced weight tensors, and
calls it does not take (strided inputs, another backend) still run."""
import pytest
import torch

from helpers import DEV, gen, q

pytestmark = pytest.mark.gpu
LIF = (1.0, 0.0, 2.0, False)


def _operands(dtype, seed=3):
    g = gen(seed)
    spikes = lambda *s: (torch.rand(*s, generator=g) < 0.3).to(DEV, dtype)
    weights = lambda *s: q(torch.randn(*s, generator=g) * 0.4, dtype).to(DEV, dtype)
    return g, spikes, weights


def _calls(dtype, zero):
    """name -> (call, weight) of every operator that the native dispatch implements, smallest shapes with a remainder."""
    S = torch.ops.snn_custom
    g, spikes, weights = _operands(dtype)
    xs = [spikes(2, 24, 7, 9) for _ in range(4)]
    rs = [spikes(2, 40, 7, 9) for _ in range(4)]
    seq = torch.randn(4, 2, 24, 7, 9, generator=g).to(DEV, dtype)
    rows = spikes(4, 5, 40)
    w3, w1, wd, b40, b24 = weights(40, 24, 3, 3), weights(40, 24, 1, 1), weights(24, 1, 3, 3), weights(40), weights(24)
    wl, bl, wt, bt = weights(33, 40), weights(33), weights(11, 24), weights(11)
    same, one = ([1, 1], [1, 1], [1, 1]), ([1, 1], [0, 0], [1, 1])
    v1 = torch.rand(2, 24, 7, 9, generator=g).to(DEV, dtype)
    return {
        "lif_forward_state": (lambda: S.lif_forward_state(xs[0], v1, *LIF), None),
        "fused_conv_lif_state": (lambda: S.fused_conv_lif_state(xs[0], w3, b40, zero, *same, 1, *LIF), w3),
        "fused_temporal_conv_lif_state": (lambda: S.fused_temporal_conv_lif_state(xs, w3, b40, zero, *same, 1, *LIF), w3),
        "fused_temporal_pointwise_conv_lif_state": (lambda: S.fused_temporal_pointwise_conv_lif_state(xs, w1, b40, zero, *one, 1, *LIF), w1),
        "fused_temporal_depthwise_conv_lif_state": (lambda: S.fused_temporal_depthwise_conv_lif_state(xs, wd, b24, zero, *same, 24, *LIF), wd),
        "fused_temporal_conv_add_lif_state": (lambda: S.fused_temporal_conv_add_lif_state(xs, rs, w3, b40, zero, *same, 1, *LIF), w3),
        "fused_temporal_lif_state": (lambda: S.fused_temporal_lif_state(seq, zero, *LIF), None),
        "fused_temporal_lif_avgpool_linear": (lambda: S.fused_temporal_lif_avgpool_linear(seq, zero, wt, bt, *LIF), wt),
        "fused_temporal_linear_lif_state": (lambda: S.fused_temporal_linear_lif_state(list(rows.unbind(0)), wl, bl, zero, *LIF), wl),
        "fused_temporal_linear_lif_state_packed": (lambda: S.fused_temporal_linear_lif_state_packed(rows, wl, None, zero, *LIF), wl),
    }


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("host_state", [False, True])
def test_known_signature_equals_first_call(hip_ops, dtype, host_state):
    from triton_snn_fusion_amd import _dispatch
    zero = torch.zeros(()) if host_state else torch.zeros((), device=DEV)
    native = _dispatch.module()
    for name, (call, weight) in _calls(dtype, zero).items():
        native.forget_plans()
        hip_ops.reset_fused_op_call_stats()
        first = call()
        once = hip_ops.get_fused_op_call_stats()
        before = sum(native.hits())
        again = [call() for _ in range(2)]
        assert name == "lif_forward_state" or sum(native.hits()) == before + 2, name      # ran natively
        for out in again:
            assert all(torch.equal(a, b) and a.dtype == b.dtype for a, b in zip(out, first)), name
        three = hip_ops.get_fused_op_call_stats()
        assert three["total"] == 3 * once["total"] and three["triton"] == 3 * once["triton"] and three["fallback"] == 0, name
        for key in ("kernel_temporal_configs", "temporal_conv_lif_runtime_by_signature"):
            assert set(three[key]) == set(once[key]), name
        assert three["kernel_temporal_configs"] == {k: 3 * n for k, n in once["kernel_temporal_configs"].items()}, name
        if weight is not None:                              # an update in place is seen by the next call
            weight.mul_(-1.0)
            flipped = call()
            hip_ops.configure_fused_op("hip", strict_triton=True, verbose=True)      # the Python implementation
            expected = call()
            hip_ops.configure_fused_op("hip", strict_triton=True)
            assert all(torch.equal(a, b) for a, b in zip(flipped, expected)), name


def test_calls_off_the_fast_path(hip_ops):
    """Strided inputs of a signature that is known contiguous, a tensor state, and the eager backend."""
    _, spikes, weights = _operands(torch.bfloat16)
    S = torch.ops.snn_custom
    zero = torch.zeros((), device=DEV)
    xs = [spikes(2, 24, 7, 9) for _ in range(3)]
    w, b = weights(40, 24, 3, 3), weights(40)
    args = (w, b, zero, [1, 1], [1, 1], [1, 1], 1, *LIF)
    ref = S.fused_temporal_conv_lif_state(xs, *args)
    S.fused_temporal_conv_lif_state(xs, *args)
    strided = [x.permute(0, 1, 3, 2).contiguous().permute(0, 1, 3, 2) for x in xs]
    out = S.fused_temporal_conv_lif_state(strided, *args)
    assert all(torch.equal(a, c) for a, c in zip(out, ref))
    two = S.fused_temporal_conv_lif_state(xs[:2], *args)
    rest = [S.fused_temporal_conv_lif_state(xs[2:], w, b, two[1], [1, 1], [1, 1], [1, 1], 1, *LIF) for _ in range(2)]
    assert all(torch.equal(a, c) for a, c in zip(rest[0], rest[1]))
    assert torch.equal(rest[0][0][0], ref[0][2]) and torch.equal(rest[0][1], ref[1])
    hip_ops.configure_fused_op("torch")
    eager = S.fused_temporal_conv_lif_state(xs, *args)
    assert hip_ops.get_fused_op_call_stats()["fallback"] == 1
    assert float((eager[0] != ref[0]).float().mean()) < 1e-2


def test_weights_of_dead_tensors_are_given_back(hip_ops):
    _, spikes, weights = _operands(torch.bfloat16)
    S = torch.ops.snn_custom
    zero = torch.zeros((), device=DEV)
    xs = [spikes(1, 8, 5, 5)]
    outs = []
    for i in range(4):                                      # the allocator hands a dead weight's address to the next one
        w, b = weights(16, 8, 3, 3), weights(16)
        outs.append(S.fused_temporal_conv_lif_state(xs, w, b, zero, [1, 1], [1, 1], [1, 1], 1, *LIF)[1])
        ref = torch.nn.functional.conv2d(xs[0].float(), w.float(), b.float(), padding=1) / 2
        fired = ref >= 1.0
        assert float((outs[-1] - torch.where(fired, torch.zeros_like(ref), ref)).abs().max()) < 1e-4   # bf16 products are exact, 73 of them added in float32: 73 * 2^-24 * |sum| < 1e-4
        del w, b


def _one_step_views(x):
    """The one step of `x` ([1, N, ...]) as contiguous tensors whose first stride is not the size of a step: the time axis moved to
    the front of a batch-first tensor, and every fourth of a sequence of four."""
    other = torch.full_like(x, 7.0)
    views = [torch.stack([x[0]], dim=1).transpose(0, 1), torch.cat([x, other, other, other])[::4]]
    for v in views:
        assert v.shape == x.shape and v.is_contiguous() and v.stride(0) != x.stride(0)
    return views


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_one_step_whose_first_stride_means_nothing(hip_ops, dtype):
    """A size-1 time axis may have any stride in a contiguous tensor: no size of anything follows from it."""
    from triton_snn_fusion_amd.runtime import hip_convlif_backend as CB
    S = torch.ops.snn_custom
    g, spikes, weights = _operands(dtype)
    zero = torch.zeros((), device=DEV)
    seq, rows = torch.randn(1, 3, 16, 5, 8, generator=g).to(DEV, dtype), spikes(1, 5, 40)
    wt, bt, wl, wc, bc = weights(11, 16), weights(11), weights(33, 40), weights(24, 16, 3, 3), weights(24)
    calls = {
        "scan": (seq, lambda x: S.fused_temporal_lif_state(x, zero, *LIF)),
        "scan from a state": (seq, lambda x: S.fused_temporal_lif_state(x, seq[0] * 0.5, *LIF)),
        "tail": (seq, lambda x: S.fused_temporal_lif_avgpool_linear(x, zero, wt, bt, *LIF)),
        "linear": (rows, lambda x: S.fused_temporal_linear_lif_state_packed(x, wl, None, zero, *LIF)),
        "convolution without a neuron": (seq, lambda x: (CB.run_hip_conv_bias_frames(x, wc, bc, [1, 1], [1, 1]),)),
        "convolution": (seq, lambda x: S.fused_temporal_conv_lif_state([x[0]], wc, bc, zero, [1, 1], [1, 1], [1, 1], 1, *LIF)),
    }
    for name, (x, call) in calls.items():
        want = call(x)
        for view in [x] + _one_step_views(x):
            for _ in range(2):
                assert all(torch.equal(a, b) for a, b in zip(call(view), want)), (name, view.stride())


@pytest.mark.parametrize("strict", [False, True])
def test_a_host_operand_next_to_gpu_operands_stays_off_the_kernels(hip_ops, strict):
    """One GPU operand brings a call to the dispatch; an input in host memory runs on the eager operators, or is refused as it is
    without the dispatch, whether or not the same call on the GPU is known."""
    hip_ops.configure_fused_op("hip", strict_triton=strict)
    S = torch.ops.snn_custom
    g = gen(8)
    host = torch.randn(3, 16, 5, 8, generator=g)
    device_zero, device_v = torch.zeros((), device=DEV), torch.rand(3, 16, 5, 8, generator=g).to(DEV)
    S.lif_forward_state(host.to(DEV), device_v, *LIF)
    want = hip_ops.lif_forward_state_torch(host, device_zero, *LIF)       # a state on another device: the step starts from zeros
    for state in (device_zero, device_v):
        got = S.lif_forward_state(host, state, *LIF)
        assert all(a.device.type == "cpu" and torch.equal(a, b) for a, b in zip(got, want))
    xs = [(torch.rand(2, 16, 5, 8, generator=g) < 0.3).float() for _ in range(4)]
    w, b = torch.randn(24, 16, 3, 3, generator=g), torch.randn(24, generator=g)
    args = ([1, 1], [1, 1], [1, 1], 1, *LIF)
    for _ in range(2):
        S.fused_temporal_conv_lif_state([x.to(DEV) for x in xs], w.to(DEV), b.to(DEV), device_zero, *args)
        S.fused_temporal_lif_state(torch.stack(xs).to(DEV), device_zero, *LIF)
    hip_ops.reset_fused_op_call_stats()
    hip_ops.configure_fused_op("hip")
    spikes, v = S.fused_temporal_lif_state(torch.stack(xs), device_zero, *LIF)
    assert spikes.device.type == v.device.type == "cpu"
    assert torch.equal(S.fused_temporal_conv_lif_state(xs, w, b, device_zero, *args)[0], S.fused_temporal_conv_lif_state(xs, w, b, torch.zeros(()), *args)[0])
    assert hip_ops.get_fused_op_call_stats()["triton"] == 0


def test_inference_weights_of_a_known_signature(hip_ops):
    """Weights made under inference mode have no version counter, so nothing is packed for them: the operators fall back (and raise in
    strict mode), the internal layouts refuse, whether or not the call is known with ordinary weights."""
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    S = torch.ops.snn_custom
    _, spikes, weights = _operands(torch.bfloat16)
    zero = torch.zeros((), device=DEV)
    xs = [spikes(2, 24, 7, 9) for _ in range(4)]
    bits = B.from_dense(torch.stack(xs))
    w, b = weights(40, 24, 3, 3), weights(40)
    with torch.inference_mode():
        wi, bi = w.clone(), b.clone()
    rest = (zero, [1, 1], [1, 1], [1, 1], 1, *LIF)
    for _ in range(2):
        S.fused_temporal_conv_lif_state(xs, w, b, *rest)
        B.conv_lif_blocked(bits, w, b, [1, 1], [1, 1], LIF[:3])
    for weight, bias in ((wi, bi), (wi, b), (w, bi)):
        for _ in range(2):
            hip_ops.configure_fused_op("hip", strict_triton=True)
            with pytest.raises(RuntimeError, match="Inference tensors"):
                S.fused_temporal_conv_lif_state(xs, weight, bias, *rest)
            with pytest.raises(RuntimeError, match="Inference tensors"):
                B.conv_lif_blocked(bits, weight, bias, [1, 1], [1, 1], LIF[:3])
            hip_ops.configure_fused_op("hip")
            hip_ops.reset_fused_op_call_stats()
            got = S.fused_temporal_conv_lif_state(xs, weight, bias, *rest)
            want = hip_ops.fused_temporal_conv_lif_state_torch(xs, weight, bias, *rest)
            assert all(torch.equal(a, c) for a, c in zip(got, want))
            assert hip_ops.get_fused_op_call_stats()["fallback"] == 1
    with torch.inference_mode():        # ordinary weights, activations that are inference tensors
        for _ in range(2):
            got = S.fused_temporal_conv_lif_state([x.clone() for x in xs], w, b, *rest)
        assert hip_ops.get_fused_op_call_stats()["triton"] == 2


@pytest.mark.parametrize("error", [torch.OutOfMemoryError, "SnnfError", KeyboardInterrupt])
def test_what_a_known_call_throws(hip_ops, monkeypatch, error):
    """An error on the native route (here: the weight cannot be packed) is answered by the Python implementation: the type of the
    exception, the counted fallback and the eager result are what they are without the dispatch. An interrupt passes through."""
    from triton_snn_fusion_amd import _dispatch, _lib
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B, hip_convlif_backend as CB, hip_temporal_linear_lif_backend as NB
    S = torch.ops.snn_custom
    _, spikes, weights = _operands(torch.bfloat16)
    zero = torch.zeros((), device=DEV)
    xs = [spikes(2, 24, 7, 9) for _ in range(4)]
    bits = B.from_dense(torch.stack(xs))
    w, b = weights(40, 24, 3, 3), weights(40)
    conv = lambda: S.fused_temporal_conv_lif_state(xs, w, b, zero, [1, 1], [1, 1], [1, 1], 1, *LIF)
    blocked = lambda: B.conv_lif_blocked(bits, w, b, [1, 1], [1, 1], LIF[:3], want_v=True)
    bias = lambda: CB.run_hip_conv_bias_frames(torch.stack(xs), w, b, [1, 1], [1, 1])
    want = conv(), blocked()[1], bias()
    eager = hip_ops.fused_temporal_conv_lif_state_torch(xs, w, b, zero, [1, 1], [1, 1], [1, 1], 1, *LIF)
    raised = (lambda: _lib.SnnfError("snnf_conv_pack_weight", -1, "planted")) if error == "SnnfError" else lambda: error("planted")
    kind = _lib.SnnfError if error == "SnnfError" else error
    tried = []

    def pack(*args):
        tried.append(args)
        raise raised()

    native = _dispatch.module()
    try:
        native.connect(hip_ops._slow_dispatch, pack, B._plane_matrix,
                       lambda device, T, M, fin, fout: NB._split_workspace(_lib.lib(), device, T, M, fin, fout))
        native.forget_weights()
        if kind is KeyboardInterrupt:
            for call in (conv, blocked, bias):
                with pytest.raises(KeyboardInterrupt):
                    call()
            assert len(tried) == 3
            return
        got = conv(), blocked()[1], bias()              # the Python implementations pack the weight
        assert len(tried) == 3 and torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
        assert all(torch.equal(a, c) for a, c in zip(got[0], want[0]))
        for module in (CB, B):
            monkeypatch.setattr(module, "_packed_weight", pack)
        for call in (conv, blocked, bias):              # strict
            with pytest.raises(kind, match="planted"):
                call()
        hip_ops.configure_fused_op("hip")
        hip_ops.reset_fused_op_call_stats()
        assert all(torch.equal(a, c) for a, c in zip(conv(), eager))
        stats = hip_ops.get_fused_op_call_stats()
        assert (stats["total"], stats["triton"], stats["fallback"]) == (1, 0, 1)
    finally:
        hip_ops.connect_native_dispatch()


def test_other_threads_run_while_a_known_call_allocates_and_launches(hip_ops):
    """With the interpreter's own switching off, another thread gets on only when a call gives the interpreter lock back."""
    import sys
    import threading
    import time
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B, hip_convlif_backend as CB, hip_pool_backend as PB
    _, spikes, weights = _operands(torch.bfloat16)
    dense = torch.stack([spikes(2, 24, 8, 8) for _ in range(4)])
    bits, half = B.from_dense(dense), B.from_dense(torch.stack([spikes(2, 48, 16, 16) for _ in range(4)]))
    x16 = B.from_dense(torch.stack([spikes(2, 32, 8, 8) for _ in range(4)]))
    w, b, wsc, bsc, w16, fc = weights(40, 24, 3, 3), weights(40), weights(40, 48, 1, 1), weights(40), weights(40, 32, 3, 3), weights(10, 24)
    one = [1, 1]
    calls = {
        "convolution": lambda: B.conv_lif_blocked(bits, w, b, one, one, LIF[:3]),
        "with a shortcut": lambda: B.conv_lif_blocked_shortcut(x16, w16, b, one, half, wsc, bsc, [2, 2], LIF[:3]),
        "with a pool": lambda: B.conv_lif_blocked_avgpool(bits, w, b, one, one, LIF[:3]),
        "pool": lambda: B.pool_blocked(bits, True, 2, 2, 0),
        "classifier": lambda: B.spike_pool_linear(bits, fc, None),
        "convolution without a neuron": lambda: CB.run_hip_conv_bias_frames(dense, w, b, one, one),
        "dense pool": lambda: PB.run_hip_pool2d(dense, True, 2, 2, 0),
    }
    progress, stop = [0], threading.Event()

    def other():
        while not stop.is_set():
            progress[0] += 1
            time.sleep(0)

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other, daemon=True)
    try:
        thread.start()
        for name, call in calls.items():
            kept = [call() for _ in range(3)]              # known, the weight packed; nothing is freed meanwhile
            sys.setswitchinterval(1000.0)
            time.sleep(0.02)                               # the other thread's next wait is one without an end
            before = progress[0]
            while progress[0] == before and len(kept) < 1000:
                kept.append(call())
            after = progress[0]
            sys.setswitchinterval(interval)
            torch.cuda.synchronize()
            assert after > before, name
    finally:
        sys.setswitchinterval(interval)
        stop.set()
        thread.join()


def test_internal_layouts_without_the_extension(hip_ops, monkeypatch):
    """The internal-layout entry points, the neuron-free convolution and the dense pool on their Python implementations alone."""
    from triton_snn_fusion_amd import _dispatch
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B, hip_convlif_backend as CB, hip_pool_backend as PB
    _, spikes, weights = _operands(torch.float16)
    dense = torch.stack([spikes(2, 24, 8, 8) for _ in range(4)])
    w, b, fc, one = weights(40, 24, 3, 3), weights(40), weights(10, 24), [1, 1]
    x = B.from_dense(dense)

    def run():
        out, v = B.conv_lif_blocked(x, w, b, one, one, LIF[:3], want_v=True)
        pooled, _ = B.conv_lif_blocked_avgpool(x, w, b, one, one, LIF[:3])
        return [out.data, v, pooled.data, B.pool_blocked(x, True, 2, 2, 0).data, B.spike_pool_linear(x, fc, None),
                CB.run_hip_conv_bias_frames(dense, w, b, one, one), PB.run_hip_pool2d(dense, True, 2, 2, 0)]

    run()
    known = run()
    monkeypatch.setattr(_dispatch, "_MODULE", _dispatch._Absent())
    assert all(torch.equal(a, c) for a, c in zip(run(), known))


def _python(call):
    """The same call through the Python implementation."""
    from triton_snn_fusion_amd import _dispatch
    native = _dispatch.module()
    native.enable(False)
    try:
        return call()
    finally:
        native.enable(True)


def _same(got, want, what):
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and torch.equal(a, b), what


def _shifted(x):
    """`x` at an odd element of its memory."""
    room = torch.empty(x.numel() + 1, device=x.device, dtype=x.dtype)
    room[1:].copy_(x.flatten())
    return room[1:].view(x.shape)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_misaligned_operands_of_a_signature_learnt_aligned(hip_ops, dtype):
    """The address is not part of a signature: the entry points look at it. Inputs, states and residuals at an odd element."""
    S = torch.ops.snn_custom
    g, spikes, weights = _operands(dtype)
    zero = torch.zeros((), device=DEV)
    xs, rs = [spikes(2, 24, 8, 8) for _ in range(4)], [spikes(2, 64, 8, 8) for _ in range(4)]
    seq, rows, v = torch.randn(4, 2, 24, 8, 8, generator=g).to(DEV, dtype), spikes(4, 8, 64), torch.rand(2, 24, 8, 8, generator=g).to(DEV, dtype)
    w3, w1, wd, b64, b24 = weights(64, 24, 3, 3), weights(64, 24, 1, 1), weights(24, 1, 3, 3), weights(64), weights(24)
    wl, bl, wt, bt = weights(32, 64), weights(32), weights(16, 24), weights(16)
    same = ([1, 1], [1, 1], [1, 1])
    calls = {
        "step": lambda m: S.lif_forward_state(m(xs[0]), m(v), *LIF),
        "scan": lambda m: S.fused_temporal_lif_state(m(seq), m(v), *LIF),
        "tail": lambda m: S.fused_temporal_lif_avgpool_linear(m(seq), m(v), m(wt), m(bt), *LIF),
        "linear": lambda m: S.fused_temporal_linear_lif_state_packed(m(rows), m(wl), m(bl), zero, *LIF),
        "linear, list": lambda m: S.fused_temporal_linear_lif_state([m(r) for r in rows.unbind(0)], m(wl), bl, zero, *LIF),
        "convolution": lambda m: S.fused_temporal_conv_add_lif_state([m(x) for x in xs], [m(r) for r in rs], w3, b64, zero, *same, 1, *LIF),
        "pointwise": lambda m: S.fused_temporal_pointwise_conv_lif_state([m(x) for x in xs], m(w1), b64, zero, [1, 1], [0, 0], [1, 1], 1, *LIF),
        "depthwise": lambda m: S.fused_temporal_depthwise_conv_lif_state([m(x) for x in xs], m(wd), m(b24), m(v), *same, 24, *LIF),
    }
    for name, call in calls.items():
        for _ in range(2):
            aligned = call(lambda t: t)
        got, want = call(_shifted), _python(lambda: call(_shifted))
        _same(got, want, name)
        if name == "tail":      # the classifier adds its 24 products in another order: 24 * 2^-24 * sum |w| count < 2e-5, or one unit of the storage
            assert torch.allclose(got[0].float(), aligned[0].float(), rtol=2.0 ** -7 if dtype == torch.bfloat16 else 0.0, atol=2e-5), name
        else:
            assert torch.equal(got[0], aligned[0]), name
    assert hip_ops.get_fused_op_call_stats()["fallback"] == 0


@pytest.mark.parametrize("state", ["zero", "tensor"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [16, 17, 33, 64, 65])
def test_long_sequences(hip_ops, T, dtype, state):
    """Windows of sixteen steps (a 16-bit membrane works in float32 between them), the most steps the dispatch takes, and one more."""
    S = torch.ops.snn_custom
    g, spikes, weights = _operands(dtype, seed=T)
    v = lambda *s: torch.rand(*s, generator=g).to(DEV, dtype) if state == "tensor" else torch.zeros(())
    seq, rows, xs = torch.randn(T, 2, 8, 5, 7, generator=g).to(DEV, dtype), spikes(T, 5, 40), [spikes(1, 8, 6, 6) for _ in range(T)]
    wl, w3, wd, b8 = weights(33, 40), weights(8, 8, 3, 3), weights(8, 1, 3, 3), weights(8)
    v5, v2, v4 = v(2, 8, 5, 7), v(5, 33), v(1, 8, 6, 6)
    same = ([1, 1], [1, 1], [1, 1])
    for name, call in {
        "scan": lambda: S.fused_temporal_lif_state(seq, v5, *LIF),
        "linear": lambda: S.fused_temporal_linear_lif_state_packed(rows, wl, None, v2, *LIF),
        "convolution": lambda: S.fused_temporal_conv_lif_state(xs, w3, b8, v4, *same, 1, *LIF),
        "depthwise": lambda: S.fused_temporal_depthwise_conv_lif_state(xs, wd, b8, v4, *same, 8, *LIF),
    }.items():
        call()
        _same(call(), _python(call), (name, T))


def test_streams_and_threads(hip_ops):
    """Known calls on streams of their own, from one thread and from four at once: scratch memory, the linear kernel's workspace (one per
    stream) and the tables of the dispatch are shared by all of them."""
    import threading
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    S = torch.ops.snn_custom
    _, spikes, weights = _operands(torch.bfloat16)
    zero = torch.zeros((), device=DEV)
    xs, rows = [spikes(8, 72, 27, 35) for _ in range(4)], spikes(4, 16, 8192)
    wc, bc, wl = weights(104, 72, 3, 3), weights(104), weights(64, 8192)
    bits = B.from_dense(torch.stack(xs))
    calls = [lambda: S.fused_temporal_conv_lif_state(xs, wc, bc, zero, [1, 1], [1, 1], [1, 1], 1, *LIF),
             lambda: S.fused_temporal_linear_lif_state_packed(rows, wl, None, zero, *LIF),
             lambda: S.lif_forward_state(xs[0], xs[1], *LIF),
             lambda: [t for t in B.conv_lif_blocked(bits, wc, bc, [1, 1], [1, 1], LIF[:3], out_layout=B.NCHW, want_v=True)]]
    plain = lambda out: [o.data if isinstance(o, B.Blocked) else o for o in out]
    for call in calls:
        call()
    want = [[t.clone() for t in plain(call())] for call in calls]
    torch.cuda.synchronize()
    wrong = []

    def work(rounds):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for _ in range(rounds):
                    outs = [plain(call()) for call in calls]
                    stream.synchronize()
                    for i, out in enumerate(outs):
                        if not all(torch.equal(a, b) for a, b in zip(out, want[i])):
                            wrong.append(i)
        except Exception as exc:                # noqa: BLE001 - reported by the assertion below
            wrong.append(repr(exc))

    work(3)
    assert not wrong, wrong
    threads = [threading.Thread(target=work, args=(20,)) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong
