"""Timed cases: what programs have this framework do, through its public entry points, over the range they use it in.

Kinds of case (`kind`):
  step      one neuron update of a single-step network: `snn_custom::lif_forward_state`
  scan      the neuron over T steps of a stack of currents: `snn_custom::fused_temporal_lif_state`
  tail      neuron over T steps, global average pool, classifier: `snn_custom::fused_temporal_lif_avgpool_linear`
  conv      convolution (+ residual) + neuron over T steps, dense tensors: `snn_custom::fused_temporal_conv_lif_state`
            and `fused_temporal_conv_add_lif_state`
  linear    linear layer + neuron over T steps: `snn_custom::fused_temporal_linear_lif_state_packed`
  block     depthwise 3x3 + neuron, pointwise 1x1 + neuron: the two operators of a depthwise-separable block
  network   a whole network: the single-step model, rewritten by `compile_temporal`, called on a batch of frames, as a plain
            call or as the replay of a HIP graph that the program captured once ("graph"), on the dense operators that the
            rewrite emits by default or on the internal layouts ("internal")

All calls are forward: the operators have no backward. Neurons are (v_th 1, v_reset 0, tau 2) throughout, spikes are
Bernoulli, weights Kaiming-normal with a gain at which a tenth of the neurons or so fires. Weights, biases and frames are
fixed-point numbers (ten bits below the weights' standard deviation, 8-bit pixels), as a quantised network has them: every sum
of a layer is then exact in float32 in any order, and no spike depends on how an implementation orders its additions.
"""
from __future__ import annotations

import math

import torch

import triton_snn_fusion_amd  # noqa: F401
from triton_snn_fusion_amd import fx_temporal_rewrite, models
from triton_snn_fusion_amd.runtime import snn_custom_ops
from triton_snn_fusion_amd.workloads import fold_bn_into_conv_params

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZES = {"bf16": 2, "f16": 2, "f32": 4}
LIF = (1.0, 0.0, 2.0)
DEVICE = "cuda:0"
GAIN = 3.0
# frame sizes, and the most frames of the largest size in one batch
NETWORK_SIZES = {"vgg11": (32, 48, 64), "resnet18": (64, 96, 128, 160, 192, 224), "mobilenet": (32, 64, 96, 128)}
MOST_FRAMES = {"vgg11": 128, "resnet18": 112, "mobilenet": 96}
CLASSES = {"vgg11": 10, "resnet18": 1000, "mobilenet": 10}


def listed():
    return [
        # one neuron layer of an eager single-step network at batch 1: pure call latency
        {"name": "step_1x64x28x28_f32", "kind": "step", "N": 1, "C": 64, "H": 28, "W": 28, "dtype": "f32"},
        # a neuron layer on a stack of currents at a streaming size (the depthwise block's plane at batch 32)
        {"name": "scan_4x32x128x56x56_bf16", "kind": "scan", "T": 4, "N": 32, "C": 128, "H": 56, "W": 56, "dtype": "bf16"},
        # the end of an ImageNet-sized classifier network
        {"name": "tail_4x16x512x7x7_k1000_bf16", "kind": "tail", "T": 4, "N": 16, "C": 512, "H": 7, "W": 7, "K": 1000, "dtype": "bf16"},
        # a single 3x3 layer on small float32 tensors: the smallest configuration of the benchmark
        {"name": "conv3x3_64_32x32_b8_f32", "kind": "conv", "T": 4, "N": 8, "Cin": 64, "Cout": 64, "H": 32, "W": 32, "k": 3, "s": 1,
         "residual": False, "membrane": "f32", "dtype": "f32"},
        # a residual layer on a plane that no tile divides, with the 16-bit membrane that the rewriter's host-side zero state selects
        {"name": "conv3x3_res_72_104_27x35_b5_f16", "kind": "conv", "T": 6, "N": 5, "Cin": 72, "Cout": 104, "H": 27, "W": 35, "k": 3, "s": 1,
         "residual": True, "membrane": "act", "dtype": "f16"},
        # the linear layer of the benchmark
        {"name": "linear_8x64_2048_1024_bf16", "kind": "linear", "T": 8, "M": 64, "Fin": 2048, "Fout": 1024, "dtype": "bf16"},
        # the depthwise-separable block of the benchmark, its two dense operators
        {"name": "block_128_256_56x56_b32_bf16", "kind": "block", "T": 4, "N": 32, "Cin": 128, "Cout": 256, "H": 56, "W": 56, "dtype": "bf16"},
        # a small classifier on one frame: the latency of a request
        {"name": "vgg11_b1_internal", "kind": "network", "net": "vgg11", "T": 4, "N": 1, "size": 32, "layouts": "internal", "launch": "eager"},
        # the CIFAR-sized network at its batch
        {"name": "vgg11_b64_internal", "kind": "network", "net": "vgg11", "T": 4, "N": 64, "size": 32, "layouts": "internal", "launch": "eager"},
        # the ImageNet-sized network at its batch on the dense operators, as the plain rewrite gives it, replayed as a graph
        {"name": "resnet18_b16_dense_graph", "kind": "network", "net": "resnet18", "T": 4, "N": 16, "size": 224, "layouts": "dense",
         "launch": "graph"},
        # the same on the internal layouts
        {"name": "resnet18_b16_internal", "kind": "network", "net": "resnet18", "T": 4, "N": 16, "size": 224, "layouts": "internal",
         "launch": "eager"},
        # throughput serving: a large batch
        {"name": "resnet18_b128_internal", "kind": "network", "net": "resnet18", "T": 4, "N": 128, "size": 224, "layouts": "internal",
         "launch": "eager"},
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _channels(rng, low, high):
    """Mostly whole groups of eight, as networks have them; any number now and then."""
    c = _spread(rng, low, high)
    return c if rng.random() < 0.2 else max(8, (c + 4) // 8 * 8)


def draw(rng):
    kind = rng.choice(["step", "scan", "tail", "conv", "conv", "linear", "block", "network", "network", "network"])
    while True:
        c = _draw(rng, kind)
        w = work(c)
        # nothing costs more than the largest listed case; a call on dense tensors stays below half a gigabyte
        if kind == "network" or (w["bytes"] <= 5e8 and w["flops"] <= 5e10):
            return c


def _draw(rng, kind):
    half = rng.choice(["bf16", "bf16", "f16"])
    any_dtype = rng.choice(["bf16", "f16", "f32"])
    T = rng.choice([1, 2, 3, 4, 4, 4, 5, 6, 8])
    if kind == "step":
        return {"kind": kind, "N": _spread(rng, 1, 64), "C": _channels(rng, 16, 512), "H": _spread(rng, 4, 56), "W": _spread(rng, 4, 56),
                "dtype": any_dtype}
    if kind == "scan":
        return {"kind": kind, "T": rng.choice([1, 4, 4, 8, 16]), "N": _spread(rng, 1, 32), "C": _channels(rng, 16, 512), "H": _spread(rng, 4, 112),
                "W": _spread(rng, 4, 112), "dtype": any_dtype}
    if kind == "tail":
        hw = _spread(rng, 1, 28)
        return {"kind": kind, "T": T, "N": _spread(rng, 1, 64), "C": _channels(rng, 64, 1024), "H": hw, "W": hw,
                "K": rng.choice([10, 100, 101, 1000]), "dtype": any_dtype}
    if kind == "conv":
        k, s = rng.choice([(3, 1), (3, 1), (3, 1), (3, 2), (1, 1), (5, 1), (7, 2)])
        h = _spread(rng, 7, 112)
        return {"kind": kind, "T": T, "N": _spread(rng, 1, 32), "Cin": _channels(rng, 16, 512), "Cout": _channels(rng, 16, 512), "H": h,
                "W": h if rng.random() < 0.6 else _spread(rng, 7, 112), "k": k, "s": s, "residual": rng.random() < 0.3,
                "membrane": rng.choice(["f32", "act"]), "dtype": rng.choice([half, half, "f32"])}
    if kind == "linear":
        return {"kind": kind, "T": T, "M": _spread(rng, 1, 256), "Fin": _spread(rng, 64, 25088) // 8 * 8 + (rng.randrange(8) if rng.random() < 0.2 else 0),
                "Fout": _spread(rng, 10, 4096), "dtype": any_dtype}
    if kind == "block":
        h = _spread(rng, 7, 112)
        return {"kind": kind, "T": T, "N": _spread(rng, 1, 32), "Cin": _channels(rng, 32, 512), "Cout": _channels(rng, 32, 512), "H": h,
                "W": h if rng.random() < 0.7 else _spread(rng, 7, 112), "dtype": half}
    net = rng.choice(["vgg11", "resnet18", "mobilenet"])
    size = rng.choice(NETWORK_SIZES[net])
    layouts = rng.choice(["dense", "internal"])
    # batches up to the one that costs about as much as the largest listed case; the dense operators take longer for a frame
    most = MOST_FRAMES[net] * (NETWORK_SIZES[net][-1] / size) ** 2 * (0.3 if layouts == "dense" else 1.0)
    N = _spread(rng, 1, min(256, int(most)))
    return {"kind": "network", "net": net, "T": rng.choice([4, 4, 4, 2, 6, 8]) if 2 * N <= most else 4, "N": N, "size": size,
            "layouts": layouts, "launch": rng.choice(["eager", "graph"])}


# ---------------------------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _grid(w, std):
    """`w` in fixed point: ten bits below the power of two at or above its standard deviation, at most eight of those."""
    e = 2.0 ** math.ceil(math.log2(std))
    return ((w * (1024.0 / e)).round() * (e / 1024.0)).clamp(-8.0 * e, 8.0 * e)


def _spikes(shape, p, g, dtype):
    return (torch.rand(shape, generator=g, device=DEVICE) < p).to(dtype)


def _weights(shape, g, dtype, gain=GAIN):
    """Kaiming-normal weights and a small bias, as a layer with its BatchNorm folded in has them."""
    std = gain * math.sqrt(2.0 / max(1, math.prod(shape[1:])))
    w = _grid(torch.randn(shape, generator=g, device=DEVICE) * std, std)
    b = _grid(torch.randn(shape[0], generator=g, device=DEVICE) * 0.1, std)
    return w.to(dtype), b.to(dtype)


def _zero(case, dtype):
    """The zero state of a first call: float32 on the device, or the host-side placeholder of rewritten graphs, which keeps the
    membrane in the activation dtype."""
    return torch.zeros(()) if case.get("membrane") == "act" else torch.zeros((), dtype=torch.float32, device=DEVICE)


def _network(case, seed):
    model = models.build_network(case["net"], seed=seed, gain=GAIN)
    with torch.no_grad():  # weights in fixed point with the BatchNorm's scale in them; the BatchNorm keeps the shift
        for m in model.modules():
            if isinstance(m, models.ConvBNNeuron):
                bn = m.bn
                w, b = fold_bn_into_conv_params(m.conv.weight, None, bn.running_mean, bn.running_var, bn.weight, bn.bias, bn.eps)
                std = float(w.std())
                m.conv.weight.copy_(_grid(w, std))
                bn.bias.copy_(_grid(b, std))
                bn.weight.fill_(1.0)
                bn.running_mean.zero_()
                bn.running_var.fill_(1.0)
                bn.eps = 0.0
    wrapper = models.SingleStepModeLoopWrapper(model, case["T"])
    gm, _ = fx_temporal_rewrite.compile_temporal(wrapper, tail_first=True, device=DEVICE, dtype=torch.bfloat16,
                                                 internal_layouts=case["layouts"] == "internal")
    return gm


def _capture(gm, frame):
    """One HIP graph of the forward, as a serving program keeps it: its input buffer, its output and the graph."""
    static = frame.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.no_grad():
        for _ in range(2):
            gm(static)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph), torch.no_grad():
        out = gm(static)
    return static, out, graph


def prepare(case, seed):
    snn_custom_ops.configure_fused_op("hip", strict_triton=False)
    g = _generator(seed)
    kind = case["kind"]
    if kind == "network":
        gm = _network(case, seed)
        pixels = torch.randint(-128, 128, (case["N"], 3, case["size"], case["size"]), generator=g, device=DEVICE)
        frame = (pixels.float() / 64.0).to(torch.bfloat16)
        state = {"kind": kind, "frame": frame, "module": gm, "graph": None}
        if case["launch"] == "graph":
            state["static"], state["out"], state["graph"] = _capture(gm, frame)
        return state
    dtype = DTYPES[case["dtype"]]
    state = {"kind": kind, "zero": _zero(case, dtype)}
    if kind == "step":
        shape = (case["N"], case["C"], case["H"], case["W"])
        state["x"] = torch.randn(shape, generator=g, device=DEVICE).to(dtype)
        state["v"] = (torch.rand(shape, generator=g, device=DEVICE) * 0.9).to(dtype)
    elif kind in ("scan", "tail"):
        state["x"] = torch.randn((case["T"], case["N"], case["C"], case["H"], case["W"]), generator=g, device=DEVICE).mul_(1.5).to(dtype)
        if kind == "tail":
            state["w"], state["b"] = _weights((case["K"], case["C"]), g, dtype, gain=1.0)
    elif kind == "linear":
        state["x"] = _spikes((case["T"], case["M"], case["Fin"]), 0.1, g, dtype)
        state["w"], state["b"] = _weights((case["Fout"], case["Fin"]), g, dtype)
    elif kind == "conv":
        x = _spikes((case["T"], case["N"], case["Cin"], case["H"], case["W"]), 0.2, g, dtype)
        state["xs"] = list(x.unbind(0))
        k, s, p = case["k"], case["s"], case["k"] // 2
        state["w"], state["b"] = _weights((case["Cout"], case["Cin"], k, k), g, dtype)
        state["geometry"] = ([s, s], [p, p], [1, 1], 1)
        state["rs"] = None
        if case["residual"]:
            ho, wo = _out(case)
            state["rs"] = list(_spikes((case["T"], case["N"], case["Cout"], ho, wo), 0.2, g, dtype).unbind(0))
    elif kind == "block":
        x = _spikes((case["T"], case["N"], case["Cin"], case["H"], case["W"]), 0.15, g, dtype)
        state["xs"] = list(x.unbind(0))
        state["dw"] = _weights((case["Cin"], 1, 3, 3), g, dtype)
        state["pw"] = _weights((case["Cout"], case["Cin"], 1, 1), g, dtype)
        state["groups"] = case["Cin"]
    return state


def run(state):
    kind = state["kind"]
    S = torch.ops.snn_custom
    if kind == "network":
        if state["graph"] is None:
            with torch.no_grad():
                return state["module"](state["frame"])
        state["static"].copy_(state["frame"])
        state["graph"].replay()
        return state["out"]
    zero = state["zero"]
    if kind == "step":
        return S.lif_forward_state(state["x"], state["v"], *LIF, False)
    if kind == "scan":
        return S.fused_temporal_lif_state(state["x"], zero, *LIF, False)
    if kind == "tail":
        return S.fused_temporal_lif_avgpool_linear(state["x"], zero, state["w"], state["b"], *LIF, False)
    if kind == "linear":
        return S.fused_temporal_linear_lif_state_packed(state["x"], state["w"], state["b"], zero, *LIF, False)
    if kind == "conv":
        if state["rs"] is None:
            return S.fused_temporal_conv_lif_state(state["xs"], state["w"], state["b"], zero, *state["geometry"], *LIF, False)
        return S.fused_temporal_conv_add_lif_state(state["xs"], state["rs"], state["w"], state["b"], zero, *state["geometry"], *LIF, False)
    hidden, v1 = S.fused_temporal_depthwise_conv_lif_state(state["xs"], *state["dw"], zero, [1, 1], [1, 1], [1, 1], state["groups"], *LIF, False)
    spikes, v2 = S.fused_temporal_pointwise_conv_lif_state(list(hidden.unbind(0)), *state["pw"], zero, [1, 1], [0, 0], [1, 1], 1, *LIF, False)
    return hidden, v1, spikes, v2


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without, and how close two correct implementations are
# ---------------------------------------------------------------------------------------------------------------
def _out(case):
    p = case["k"] // 2
    return (case["H"] + 2 * p - case["k"]) // case["s"] + 1, (case["W"] + 2 * p - case["k"]) // case["s"] + 1


def _conv_layers(case):
    """(steps, Cin, Cout, k, groups, output pixels) of every convolution of a network. The first layer's input is the same frame
    at every step: one step's products are enough."""
    h, T, first = case["size"], case["T"], True
    if case["net"] == "vgg11":
        cin, size = 3, h
        for i, stage in enumerate(models.VGG11_STAGES):
            size = size // 2 if i else size
            for c in stage:
                yield (1 if first else T), cin, c, 3, 1, size * size
                cin, first = c, False
    elif case["net"] == "resnet18":
        size = (h + 1) // 2
        yield 1, 3, 64, 7, 1, size * size
        size, cin = (size + 1) // 2, 64
        for i in range(4):
            c = 64 << i
            if i:
                size = (size + 1) // 2
                yield T, cin, c, 1, 1, size * size
            yield T, cin, c, 3, 1, size * size
            for _ in range(3):
                yield T, c, c, 3, 1, size * size
            cin = c
    else:
        size = (h + 1) // 2
        yield 1, 3, 32, 3, 1, size * size
        cin = 32
        for c, stride in models.MOBILENET_BLOCKS:
            size = (size + stride - 1) // stride
            yield T, cin, cin, 3, cin, size * size
            yield T, cin, c, 1, 1, size * size
            cin = c


def work(case):
    kind = case["kind"]
    if kind == "network":
        flops, weights, last = 0, 0, 0
        for steps, cin, cout, k, groups, pixels in _conv_layers(case):
            flops += 2 * steps * case["N"] * pixels * cout * (cin // groups) * k * k
            weights += cout * (cin // groups) * k * k + cout
            last = cout
        classes = CLASSES[case["net"]]
        weights += classes * (last + 1)
        flops += 2 * case["N"] * classes * last
        return {"bytes": 2 * (case["N"] * 3 * case["size"] ** 2 + weights + case["N"] * classes), "flops": flops}
    b = SIZES[case["dtype"]]
    if kind == "linear":
        T, M, fin, fout = case["T"], case["M"], case["Fin"], case["Fout"]
        return {"bytes": b * (T * M * fin + fout * fin + fout + T * M * fout) + 4 * M * fout, "flops": 2 * T * M * fin * fout}
    N, plane = case["N"], case["H"] * case["W"]
    if kind == "step":
        n = N * case["C"] * plane
        return {"bytes": 4 * n * b, "flops": 4 * n}
    if kind == "scan":
        n = N * case["C"] * plane
        return {"bytes": 2 * case["T"] * n * b + 4 * n, "flops": 4 * case["T"] * n}
    if kind == "tail":
        n = N * case["C"] * plane
        return {"bytes": case["T"] * n * b + 4 * n + b * (case["K"] * (case["C"] + 1) + N * case["K"]),
                "flops": 4 * case["T"] * n + 2 * N * case["C"] * case["K"]}
    T, cin, cout = case["T"], case["Cin"], case["Cout"]
    if kind == "block":
        n = N * plane
        return {"bytes": n * (T * b * (2 * cin + cout) + 4 * (cin + cout)) + b * (9 * cin + cin * cout + cin + cout),
                "flops": 2 * T * n * (9 * cin + cin * cout)}
    ho, wo = _out(case)
    out = N * cout * ho * wo
    vb = b if case["membrane"] == "act" else 4
    steps = 2 if case["residual"] else 1
    return {"bytes": b * (T * N * cin * plane + cout * cin * case["k"] ** 2 + cout + steps * T * out) + vb * out,
            "flops": 2 * T * out * cin * case["k"] ** 2}


def tolerance(case):
    """Spikes are exact (see the top of this file). Membranes and logits carry the rounding of their dtype: float32 sums 1e-5,
    16-bit results 1e-2."""
    kind = case["kind"]
    if kind == "network":
        return {"rel": 1e-2, "max": 5e-2}
    wide = kind in ("scan", "linear", "block") or case.get("membrane") == "f32" or case["dtype"] == "f32"
    return {"rel": 1e-5, "max": 1e-4} if wide and kind != "tail" or case["dtype"] == "f32" else {"rel": 1e-2, "max": 5e-2}
