"""The work this library is used for, as timed cases: quantized networks run through GpuNet and through the C++ Frame_HIP
cells, quantization-aware learning through the Frame_HIP_QAT cells, and the float passes of single learning layers through
the C ABI.

Four kinds of case:

  infer   a batch of byte images that is on the GPU -> logits: GpuNet's graph-edge conversion and forward, launched cell by
          cell ("eager") or replayed from the HIP graph that GpuNet.capture() recorded ("graph")
  cells   the same networks as N2D2 drives them: float stimuli in host memory in, float outputs in host memory out
          (frame_hip.Net: set_stimuli, propagate, outputs)
  learn   learning iterations of a whole net of float cells with SAT quantizers (frame_hip.TrainNet.learn), then what a
          program reads of it: the loss, the weights, the BatchNorm parameters, the quantizers' alphas
  layer   one convolution layer of a learning net through the C ABI, its forward pass (weight quantizer, convolution,
          BatchNorm, activation quantizer) or its backward pass (activation quantizer, BatchNorm, both convolution
          gradients, weight quantizer, SGD), on the tensors a learning program keeps from pass to pass

Network sizes are those of the benchmark configurations (n2d2_amd/nets.py) and of the learning tests.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

from n2d2_amd import capi, frame_hip, nets, runtime

NETS = {"lenet": nets.lenet, "mobilenet_v1": nets.mobilenet_v1, "resnet50": nets.resnet50, "resnet18_w4a4": nets.resnet18_w4a4}


def listed():
    return [
        # one digit image, the smallest call: what a device that classifies one input at a time waits for
        {"name": "lenet one image", "kind": "infer", "net": "lenet", "batch": 1, "image": 32, "launch": "graph"},
        # the benchmark's LeNet batch, cell by cell: a program without a graph, where the host's launches count
        {"name": "lenet 256 eager", "kind": "infer", "net": "lenet", "batch": 256, "image": 32, "launch": "eager"},
        # one camera frame through the mobile network, depthwise and pointwise layers with few pixels each
        {"name": "mobilenet one image", "kind": "infer", "net": "mobilenet_v1", "batch": 1, "image": 224, "launch": "graph"},
        # the benchmark's MobileNet batch: throughput serving
        {"name": "mobilenet 64", "kind": "infer", "net": "mobilenet_v1", "batch": 64, "image": 224, "launch": "graph"},
        # the headline: offline classification in large batches
        {"name": "resnet50 128", "kind": "infer", "net": "resnet50", "batch": 128, "image": 224, "launch": "graph"},
        # a request queue that is not full, images of another size: odd batch, ragged rows in every layer
        {"name": "resnet50 5 of 193", "kind": "infer", "net": "resnet50", "batch": 5, "image": 193, "launch": "eager"},
        # N2D2's own call path with 4-bit weights and activations: float images in host memory in, logits in host memory out
        {"name": "resnet18 w4a4 cells 16", "kind": "cells", "net": "resnet18_w4a4", "batch": 16, "image": 224},
        # learning the small network the reference's quantization-aware test trains, small batch, 4-bit activations
        {"name": "learn lenet 32", "kind": "learn", "net": "lenet_bn", "batch": 32, "channels": 6, "size": 32, "bits": 4, "iterations": 10},
        # learning a residual block on images of CIFAR's size
        {"name": "learn residual 64", "kind": "learn", "net": "residual", "batch": 64, "channels": 64, "size": 32, "bits": 4, "iterations": 1},
        # the benchmark's learning layer (ResNet-18's first stage), forward
        {"name": "layer 64x56 forward", "kind": "layer", "pass": "forward", "quant": "sat", "bits": 4, "batch": 64, "channels": 64, "outputs": 64,
         "kernel": 3, "stride": 1, "height": 56, "width": 56, "depthwise": False},
        # a layer between two stages: stride 2, odd image and batch, step sizes learnt, backward
        {"name": "layer 128 to 256 backward", "kind": "layer", "pass": "backward", "quant": "lsq", "bits": 8, "batch": 33, "channels": 128,
         "outputs": 256, "kernel": 3, "stride": 2, "height": 27, "width": 27, "depthwise": False},
        # MobileNet's depthwise layer at 56 x 56, backward
        {"name": "layer depthwise backward", "kind": "layer", "pass": "backward", "quant": "sat", "bits": 8, "batch": 32, "channels": 128,
         "outputs": 128, "kernel": 3, "stride": 1, "height": 56, "width": 56, "depthwise": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["infer", "cells", "learn", "layer"], weights=[6, 1, 2, 5])[0]
    if kind in ("infer", "cells"):
        net = rng.choice(sorted(NETS))
        case = {"kind": kind, "net": net, "batch": _log_int(rng, 1, (256 if net == "lenet" else 128) if kind == "infer" else 32),
                "image": 32 if net == "lenet" else rng.randint(64, 224)}
        if kind == "infer":
            case["launch"] = rng.choice(["graph", "eager"])
        return case
    if kind == "learn":
        net = rng.choice(["lenet_bn", "residual"])
        lenet = net == "lenet_bn"
        return {"kind": kind, "net": net, "batch": _log_int(rng, 2, 256 if lenet else 64), "channels": 6 if lenet else _log_int(rng, 8, 96),
                "size": 32 if lenet else rng.randint(8, 32), "bits": rng.choice([4, 8]), "iterations": rng.randint(1, 10) if lenet else rng.randint(1, 2)}
    depthwise = rng.random() < 0.25
    k = rng.choice([1, 3, 3, 3, 5])
    if depthwise and k == 1:
        k = 3
    ch = _log_int(rng, 8, 512)
    case = {"kind": kind, "pass": rng.choice(["forward", "backward"]), "quant": rng.choice(["sat", "lsq"]), "bits": rng.choice([4, 8]), "batch": _log_int(rng, 1, 128),
            "channels": ch, "outputs": ch if depthwise else _log_int(rng, 8, 512), "kernel": k, "stride": rng.choice([1, 1, 2]),
            "height": _log_int(rng, 7, 112), "width": _log_int(rng, 7, 112), "depthwise": depthwise}
    # at most about the arithmetic of a ResNet stage at batch 64, and tensors of at most 128 MiB
    while case["batch"] > 1 and (work(case)["flops"] > 6e10 or case["batch"] * max(case["channels"], case["outputs"]) * case["height"] * case["width"] > 1 << 25):
        case["batch"] = case["batch"] // 2
    return case


# ------------------------------------------------------------------------------------------- quantized networks

@functools.lru_cache(maxsize=None)
def _spec(net, image):
    """The network's description: weights and rescales as post-training quantization leaves them (one network whatever the
    inputs are; calibrating it is not part of running it)."""
    return NETS[net]() if net == "lenet" else NETS[net](image=image)


def _images(case, seed):
    shape = (case["batch"],) + tuple(_spec(case["net"], case["image"]).in_shape)
    return np.random.default_rng(seed).integers(0, 256, size=shape, dtype=np.uint8)


def _prepare_infer(case, seed):
    net = nets.GpuNet(_spec(case["net"], case["image"]), case["batch"])
    net.set_input(_images(case, seed))
    state = {"case": case, "net": net}
    if case["launch"] == "graph":
        state["replay"] = net.capture(1, with_input_conversion=True)
    return state


def _run_infer(state):
    net = state["net"]
    if "replay" in state:
        out = state["replay"]()
    else:
        net.convert_input()
        out = net.forward()
    return out.buf.view(out.B, out.cs)[:, :out.C]


def _prepare_cells(case, seed):
    # 8-bit export with unsigned data and unsigned stimuli: the state N2D2's quantization pass leaves
    frame_hip.set_globals(8, True, True)
    spec = _spec(case["net"], case["image"])
    net = frame_hip.build_net(spec, case["batch"])
    net.initialize()
    return {"case": case, "net": net, "x": _images(case, seed).astype(np.float32), "output": spec.output}


def _run_cells(state):
    net = state["net"]
    net.set_stimuli(state["x"])
    net.propagate()
    return net.outputs(state["output"])


# ------------------------------------------------------------------------------------------- learning a whole net

def _weights(rng, *shape):
    return (rng.standard_normal(shape) * math.sqrt(2.0 / math.prod(shape[1:]))).astype(np.float32)


def _residual_fc_inputs(case):
    return case["channels"] * (case["size"] // 2) ** 2


def _prepare_learn(case, seed):
    rng = np.random.default_rng(seed)
    B, R = case["batch"], (1 << case["bits"]) - 1
    lenet = case["net"] == "lenet_bn"
    x = rng.random((B, 1 if lenet else 3, case["size"], case["size"]), dtype=np.float32)
    net = frame_hip.TrainNet(x, propagate_gradient=False)
    convs, bns, quants, fcs = [], [], [], []

    def conv(name, O, Cn, k, pad=0, w_range=R):
        net.add_conv(name, _weights(rng, O, Cn, k, k), pad=(pad, pad), act="Linear", weight_quant="SAT", weight_range=w_range)
        convs.append(name)

    def batchnorm(name, quant=True):
        if quant:
            net.add_batchnorm(name, act="Linear", act_quant="SAT", act_range=R, act_param=2.5)
            quants.append(name)
        else:
            net.add_batchnorm(name)
        bns.append(name)

    def fc(name, O, K, quant_range):
        net.add_fc(name, _weights(rng, O, K), act="Linear", act_quant="SAT", act_range=quant_range, act_param=4.0, weight_quant="SAT", weight_range=R,
                   apply_scaling=True)
        fcs.append(name)
        quants.append(name)

    if lenet:
        conv("conv1", 6, 1, 5, w_range=255)
        batchnorm("bn1")
        net.add_pool("pool1", (2, 2), (2, 2))
        conv("conv2", 16, 6, 5)
        batchnorm("bn2")
        net.add_pool("pool2", (2, 2), (2, 2))
        conv("conv3", 120, 16, 5)
        batchnorm("bn3")
        fc("fc1", 84, 120, R)
        fc("fc2", 10, 84, 255)
    else:
        ch = case["channels"]
        conv("stem", ch, 3, 3, 1, w_range=255)
        batchnorm("stem_bn")
        conv("a", ch, ch, 3, 1)
        batchnorm("a_bn")
        conv("b", ch, ch, 3, 1)
        batchnorm("b_bn", quant=False)
        net.add_elemwise("sum", ["b_bn", "stem_bn"], act="Linear", act_quant="SAT", act_range=R, act_param=3.0)
        quants.append("sum")
        net.add_pool("pool", (2, 2), (2, 2))
        fc("fc", 10, _residual_fc_inputs(case), 255)
    net.add_softmax("softmax")
    for name in convs + fcs:
        net.set_solver_parameter(name, "Momentum", 0.9)
    targets = np.zeros((B, 10, 1, 1), dtype=np.float32)
    targets[np.arange(B), rng.integers(0, 10, size=B)] = 1.0
    return {"case": case, "net": net, "targets": targets, "weights": convs + fcs, "bns": bns, "quants": quants}


def _run_learn(state):
    net = state["net"]
    out = {"loss": net.learn(state["targets"], state["case"]["iterations"])}
    for name in state["weights"]:
        out[name] = net.weights(name)
    for name in state["bns"]:
        p = net.batchnorm(name)
        out[name] = [p["scales"], p["biases"], p["means"], p["variances"]]
    out["alphas"] = np.array([net.activation_quantizer(name)[0] for name in state["quants"]], dtype=np.float32)
    return out


# ------------------------------------------------------------------------------------------- one learning layer

def _layer_dims(case):
    k, s = case["kernel"], case["stride"]
    pad = k // 2
    oH, oW = ((case[d] + 2 * pad - k + s) // s for d in ("height", "width"))
    return pad, oH, oW


def _prepare_layer(case, seed):
    lib = capi.lib
    B, Cn, O, k, H, W = (case[n] for n in ("batch", "channels", "outputs", "kernel", "height", "width"))
    pad, oH, oW = _layer_dims(case)
    groups = Cn if case["depthwise"] else 1
    gen = torch.Generator(device="cuda").manual_seed(seed)
    f32 = dict(dtype=torch.float32, device="cuda")
    R = (1 << case["bits"]) - 1
    s = {"case": case, "R": R, "desc": capi.ConvDesc(Cn, O, k, k, case["stride"], case["stride"], pad, pad, pad, pad, 1, 1, groups, 0)}
    vec = lambda v: torch.full((O,), v, **f32)  # noqa: E731
    # the layer's input is the fake-quantized output of the layer before: levels between 0 and alpha, half of them 0
    s["x"] = torch.clamp(torch.randn(B, Cn, H, W, generator=gen, **f32), 0.0, 2.5).mul_(R / 2.5).round_().mul_(2.5 / R)
    s["w"] = torch.randn(O, Cn // groups, k, k, generator=gen, **f32) * math.sqrt(2.0 / (Cn // groups * k * k))
    s["wq"], s["stats"] = torch.empty_like(s["w"]), torch.zeros(2, **f32)
    # weights: signed levels; step size as LSQ initialises it, 2 mean|w| / sqrt(largest level)
    s["w_lo"], s["w_hi"] = -((R + 1) // 2), (R - 1) // 2
    s["w_step"] = (2.0 * s["w"].abs().mean() / math.sqrt(max(s["w_hi"], 1))).reshape(1)
    s["alpha"], s["a_step"] = torch.full((1,), 2.5, **f32), torch.full((1,), 2.5 / R, **f32)
    s["scale"], s["bias"], s["mean"], s["var"] = vec(1.0), vec(0.0), vec(0.0), vec(1.0)
    s["smean"], s["svar"] = vec(0.0), vec(0.0)
    s["y"] = torch.empty(B, O, oH, oW, **f32)
    s["z"], s["fp"] = torch.empty_like(s["y"]), torch.empty_like(s["y"])
    n, nw = s["y"].numel(), s["w"].numel()
    s["conv_ws"] = torch.empty(max(int(lib.n2d2hip_conv2d_f32_workspace_bytes(C.byref(s["desc"]), B, H, W)), 4), dtype=torch.uint8, device="cuda")
    s["bn_ws"] = torch.empty(int(lib.n2d2hip_batchnorm_f32_workspace_bytes(B, O, oH, oW)), dtype=torch.uint8, device="cuda")
    s["q_ws"] = torch.empty(int(lib.n2d2hip_quantizer_workspace_bytes(max(n, nw))), dtype=torch.uint8, device="cuda")
    if case["pass"] == "backward":
        # what the forward pass of the same iteration left, and the gradient that comes from the layer behind
        s["y"].normal_(0.0, 3.0, generator=gen)
        s["smean"].copy_(s["y"].mean(dim=(0, 2, 3)))
        s["svar"].copy_(s["y"].var(dim=(0, 2, 3), unbiased=False) if B * oH * oW > 1 else vec(1.0))
        s["fp"].copy_((s["y"] - s["smean"][:, None, None]) / torch.sqrt(s["svar"][:, None, None] + 1e-5))
        s["dz"] = torch.randn(B, O, oH, oW, generator=gen, **f32) * 1e-3
        s["wq"].copy_(s["w"])
        s["stats"].copy_(torch.stack([torch.tanh(s["w"]).abs().max(), torch.ones((), **f32)]))
        s["g"], s["dx"] = torch.empty_like(s["y"]), torch.empty_like(s["x"])
        s["dwq"], s["dw"], s["momentum"] = torch.empty_like(s["w"]), torch.empty_like(s["w"]), torch.zeros_like(s["w"])
        s["dstep"], s["dalpha"] = torch.zeros(1, **f32), torch.zeros(1, **f32)
        s["dscale"], s["dbias"], s["dsm"], s["dsv"] = vec(0.0), vec(0.0), vec(0.0), vec(0.0)
    return s


def _run_forward(s):
    case, lib, chk, st = s["case"], capi.lib, capi.check, runtime.stream_ptr()
    B, H, W, O = case["batch"], case["height"], case["width"], case["outputs"]
    _, oH, oW = _layer_dims(case)
    p = lambda n: s[n].data_ptr()  # noqa: E731
    n, nw = s["y"].numel(), s["w"].numel()
    sat = case["quant"] == "sat"
    if sat:
        chk(lib.n2d2hip_sat_weight_forward(p("w"), p("wq"), nw, float(s["R"]), capi.SAT_DEFAULT, 0, 1, p("stats"), p("q_ws"), s["q_ws"].numel(), st))
    else:
        chk(lib.n2d2hip_lsq_forward(p("w"), p("wq"), nw, p("w_step"), s["w_lo"], s["w_hi"], st))
    chk(lib.n2d2hip_conv2d_f32_forward(C.byref(s["desc"]), B, H, W, p("x"), p("wq"), None, 0.0, p("y"), p("conv_ws"), s["conv_ws"].numel(), st))
    chk(lib.n2d2hip_batchnorm_f32_forward(B, O, oH, oW, p("y"), p("scale"), p("bias"), p("mean"), p("var"), p("smean"), p("svar"), 1e-5, 0.1, 0,
                                          p("z") if sat else p("fp"), p("bn_ws"), s["bn_ws"].numel(), st))
    if sat:
        chk(lib.n2d2hip_sat_act_forward(p("z"), p("fp"), n, float(s["R"]), p("alpha"), st))
    else:
        chk(lib.n2d2hip_lsq_forward(p("fp"), p("z"), n, p("a_step"), 0, s["R"], st))
    return {k: s[k] for k in ("wq", "y", "fp", "z", "mean", "var", "smean", "svar")}


def _run_backward(s):
    case, lib, chk, st = s["case"], capi.lib, capi.check, runtime.stream_ptr()
    B, H, W, O = case["batch"], case["height"], case["width"], case["outputs"]
    _, oH, oW = _layer_dims(case)
    p = lambda n: s[n].data_ptr()  # noqa: E731
    n, nw, R = s["y"].numel(), s["w"].numel(), s["R"]
    sat, q_ws, rate = case["quant"] == "sat", s["q_ws"].numel(), 0.01 / B
    if sat:
        chk(lib.n2d2hip_sat_act_backward(p("dz"), p("fp"), p("g"), n, float(R), p("alpha"), 0.0, p("dalpha"), p("q_ws"), q_ws, st))
    else:
        chk(lib.n2d2hip_lsq_backward(p("dz"), p("fp"), p("g"), n, p("a_step"), 0, R, 1.0 / math.sqrt(float(n) * R), 0.0, p("dalpha"), p("q_ws"), q_ws, st))
    chk(lib.n2d2hip_batchnorm_f32_backward(B, O, oH, oW, p("y"), p("scale"), p("smean"), p("svar"), 1e-5, p("g"), 0.0, p("dscale"), 0.0, p("dbias"),
                                           p("dsm"), p("dsv"), p("g"), p("bn_ws"), s["bn_ws"].numel(), st))
    d, ws = C.byref(s["desc"]), s["conv_ws"].numel()
    chk(lib.n2d2hip_conv2d_f32_backward_filter(d, B, H, W, p("x"), p("g"), 0.0, p("dwq"), p("conv_ws"), ws, st))
    chk(lib.n2d2hip_conv2d_f32_backward_data(d, B, H, W, p("wq"), p("g"), 0.0, p("dx"), p("conv_ws"), ws, st))
    if sat:
        chk(lib.n2d2hip_sat_weight_backward(p("dwq"), p("w"), p("dw"), nw, float(R), capi.SAT_DEFAULT, 0, p("stats"), st))
    else:
        chk(lib.n2d2hip_lsq_backward(p("dwq"), p("w"), p("dw"), nw, p("w_step"), s["w_lo"], s["w_hi"], 1.0 / math.sqrt(float(nw) * max(s["w_hi"], 1)), 0.0,
                                     p("dstep"), p("q_ws"), q_ws, st))
    chk(lib.n2d2hip_sgd_update_f32(p("w"), p("dw"), nw, rate, 0.9, rate * 1e-4, p("momentum"), 0, 0.0, 0.0, st))
    chk(lib.n2d2hip_sgd_update_f32(p("scale"), p("dscale"), O, rate, 0.0, 0.0, None, 0, 0.0, 0.0, st))
    chk(lib.n2d2hip_sgd_update_f32(p("bias"), p("dbias"), O, rate, 0.0, 0.0, None, 0, 0.0, 0.0, st))
    chk(lib.n2d2hip_sgd_update_f32(p("alpha") if sat else p("a_step"), p("dalpha"), 1, rate, 0.0, 0.0, None, 0, 0.0, 0.0, st))
    return {k: s[k] for k in ("g", "dx", "dwq", "dw", "w", "momentum", "dscale", "dbias", "scale", "bias", "dalpha", "alpha" if sat else "a_step")}


# ------------------------------------------------------------------------------------------- what is asked of this file

def prepare(case, seed):
    return {"infer": _prepare_infer, "cells": _prepare_cells, "learn": _prepare_learn, "layer": _prepare_layer}[case["kind"]](case, seed)


def run(state):
    kind = state["case"]["kind"]
    if kind == "layer":
        return (_run_forward if state["case"]["pass"] == "forward" else _run_backward)(state)
    return {"infer": _run_infer, "cells": _run_cells, "learn": _run_learn}[kind](state)


def work(case):
    kind, B = case["kind"], case["batch"]
    if kind in ("infer", "cells"):
        spec = _spec(case["net"], case["image"])
        weights = sum(l.w.size // (2 if l.weight_bits == 4 else 1) for l in spec.layers if l.type in ("conv", "fc"))
        values = B * (math.prod(spec.in_shape) * (1 if kind == "infer" else 4) + 4 * math.prod(spec.shapes[spec.output]))
        return {"bytes": weights + values, "flops": 2 * B * spec.macs_per_image()}
    if kind == "learn":
        if case["net"] == "lenet_bn":
            macs, n_weights, x = 28 * 28 * 150 + 10 * 10 * 2400 + 48000 + 84 * 120 + 840, 150 + 2400 + 48000 + 84 * 120 + 840, 1024
        else:
            ch, hw = case["channels"], case["size"] ** 2
            n_weights, x = 27 * ch + 18 * ch * ch + 10 * _residual_fc_inputs(case), 3 * hw
            macs = hw * (27 * ch + 18 * ch * ch) + 10 * _residual_fc_inputs(case)
        # the images and targets and, in and out, weights and momentum of an iteration; three products of a layer's size
        return {"bytes": 4 * case["iterations"] * (B * (x + 10) + 4 * n_weights), "flops": 6 * case["iterations"] * B * macs}
    _, oH, oW = _layer_dims(case)
    per_output = (1 if case["depthwise"] else case["channels"]) * case["kernel"] ** 2
    nx, ny, nw = B * case["channels"] * case["height"] * case["width"], B * case["outputs"] * oH * oW, case["outputs"] * per_output
    if case["pass"] == "forward":       # x, w in; quantized weights, y, fp and z out
        return {"bytes": 4 * (nx + 2 * nw + 3 * ny), "flops": 2 * ny * per_output}
    # x, dz, fp, y, both weights and the momentum in; the gradients of y, x and both weights, weights and momentum out
    return {"bytes": 4 * (2 * nx + 4 * ny + 7 * nw), "flops": 4 * ny * per_output}


def tolerance(case):
    if case["kind"] in ("infer", "cells"):
        return "exact"              # integers
    if case["kind"] == "learn":
        # activations are numbers of 4 to 8 bits inside: a 32-bit sum that differs in its last bits moves a value over a
        # rounding edge here and there, and the gradients of the parameters with it
        return {"rel": 5e-3, "max": 0.2}
    if case["pass"] == "forward":
        # the fake-quantized output holds levels of alpha / (2^bits - 1): for a value on an edge one level is the step
        return {"rel": 1e-3, "max": 0.9}
    return {"rel": 2e-5}            # 32-bit sums throughout
