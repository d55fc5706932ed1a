"""The calls that a program using this package makes, as cases to be timed.

Three paths through the public classes:

* ``layer``: one pruned 1x1 convolution (``SparseConvKernel.Run``) in fp32,
  fp16, int8 -> fp32 or int8 -> int8;
* ``quantised``: an int8 layer in an fp32 program: the activations go through
  ``CalibComputeFp32ToInt8`` and the layer hands back fp32;
* ``body``: the convolutional body of MobileNetV1-1.0 in int8, thirteen times a
  depthwise 3x3 and a pruned 1x1 layer, each consuming the output of the one
  before; a 1x1 layer and the depthwise layer behind it run as one launch
  where the library says that this pays.

Shapes are those of the benchmark configurations and of the benchmark's
floating-point layers.
"""
import importlib

import numpy as np
import torch

pla = importlib.import_module("paddle-lite_amd")
capi = pla.capi
workloads = importlib.import_module("paddle-lite_amd.workloads")
depthwise = importlib.import_module("paddle-lite_amd.depthwise_conv")

PRECISIONS = {"fp32": ("float32", "float32"), "fp16": ("float16", "float16"), "int8_fp32": ("int8", "float32"), "int8_int8": ("int8", "int8")}
IN_BYTES = {"fp32": 4, "fp16": 2, "int8_fp32": 1, "int8_int8": 1}
OUT_BYTES = {"fp32": 4, "fp16": 2, "int8_fp32": 4, "int8_int8": 1}
ACTIVATIONS = ["none", "relu", "relu6", "leaky_relu", "hard_swish"]


def _layer(name, kind, batch, ic, oc, h, w, sparsity, pairs, act):
    return {"name": name, "path": "layer", "kind": kind, "batch": batch, "ic": ic, "oc": oc, "h": h, "w": w, "sparsity": sparsity, "pairs": pairs, "act": act}


def listed():
    return [
        # one image through one fp32 layer on a device that is otherwise idle: latency
        _layer("fp32_96_192_56_one_image", "fp32", 1, 96, 192, 56, 56, 0.80, False, "relu"),
        # a batch through a layer pruned in pairs of output channels
        _layer("fp32_pairs_256_512_28", "fp32", 32, 256, 512, 28, 28, 0.90, True, "relu6"),
        # the deep layers of a network, pruned weight by weight
        _layer("fp32_512_512_14", "fp32", 64, 512, 512, 14, 14, 0.85, False, "relu"),
        # the last layers of a network: many channels, maps of 49 positions
        _layer("fp32_pairs_1024_1024_7", "fp32", 64, 1024, 1024, 7, 7, 0.70, True, "relu"),
        # half precision, one deep layer on maps that are a multiple of 4 positions only, one on odd maps
        _layer("fp16_512_512_14", "fp16", 64, 512, 512, 14, 14, 0.85, False, "relu"),
        _layer("fp16_pairs_128_256_55", "fp16", 8, 128, 256, 55, 55, 0.70, True, "relu"),
        # the headline configuration
        _layer("int8_fp32_512_512_14", "int8_fp32", 64, 512, 512, 14, 14, 0.85, False, "leaky_relu"),
        # the largest single layer: requantised output with the costly activation
        _layer("int8_int8_pairs_128_256_56", "int8_int8", 128, 128, 256, 56, 56, 0.75, True, "hard_swish"),
        # a wide layer: more channels than a workgroup holds at once
        _layer("int8_fp32_2048_2048_14", "int8_fp32", 16, 2048, 2048, 14, 14, 0.90, False, "leaky_relu"),
        # an int8 layer between fp32 ones, odd maps
        {"name": "quantised_192_384_17", "path": "quantised", "kind": "int8_fp32", "batch": 64, "ic": 192, "oc": 384, "h": 17, "w": 17, "sparsity": 0.85, "pairs": False, "act": "relu6"},
        # a whole network body, one image (latency) and a batch (throughput)
        {"name": "mobilenet_v1_body_one_image", "path": "body", "batch": 1, "sparsity": 0.90},
        {"name": "mobilenet_v1_body_64", "path": "body", "batch": 64, "sparsity": 0.90},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(float(lo) * (float(hi) / lo) ** rng.random()))


def _channels(rng):
    """32 .. 2048, mostly the multiples of 32 that networks use, sometimes any number."""
    c = _log_uniform(rng, 32, 2048)
    return c if rng.random() < 0.3 else max(32, c // 32 * 32)


def draw(rng):
    if rng.random() < 0.15:
        return {"path": "body", "batch": _log_uniform(rng, 1, 48), "sparsity": round(rng.uniform(0.7, 0.95), 2)}
    quantised = rng.random() < 0.15
    kind = "int8_fp32" if quantised else rng.choice(["fp32", "fp16", "int8_fp32", "int8_int8"])
    while True:
        side = _log_uniform(rng, 7, 112)
        case = {"path": "quantised" if quantised else "layer", "kind": kind, "batch": _log_uniform(rng, 1, 128), "ic": _channels(rng), "oc": _channels(rng), "h": side,
                "w": side if rng.random() < 0.7 else max(7, side + rng.randint(-5, 5)), "sparsity": round(rng.uniform(0.7, 0.95), 2), "pairs": rng.random() < 0.4, "act": rng.choice(ACTIVATIONS)}
        cost = work(case)
        if cost["bytes"] <= 150e6 and cost["flops"] <= (1.5e9 if kind in ("fp32", "fp16") else 5e9):
            return case


def _activation(act):
    if act == "none":
        return pla.ActivationParam()
    if act == "leaky_relu":
        return pla.ActivationParam("leaky_relu", Leaky_relu_alpha=0.1)
    return pla.ActivationParam(act)


def _conv(case, seed):
    """The prepared kernel of one pruned layer: weights and bias from the seed, output scale of an int8 output at
    three standard deviations of its values."""
    rng = np.random.RandomState(seed % 2**32)
    oc, ic = case["oc"], case["ic"]
    if case["pairs"]:
        keep = np.repeat(rng.random_sample(((oc + 1) // 2, ic)) >= case["sparsity"], 2, axis=0)[:oc]
    else:
        keep = rng.random_sample((oc, ic)) >= case["sparsity"]
    bias = (rng.standard_normal(oc) * 0.1).astype(np.float32)
    if case["kind"] in ("fp32", "fp16"):
        dense = (rng.standard_normal((oc, ic)) * 0.1).astype(np.float32) * keep
        param = dict(enable_int8=False)
    else:
        dense = (rng.randint(1, 128, size=(oc, ic)) * (rng.randint(0, 2, size=(oc, ic)) * 2 - 1) * keep).astype(np.int8)
        weight_scale = rng.uniform(0.001, 0.02, size=oc).astype(np.float32)
        sigma = np.sqrt(ic * (1.0 - case["sparsity"])) * 73.3 * 73.3 * float(weight_scale.mean()) * 0.01
        param = dict(enable_int8=True, input_scale=0.01, weight_scale=weight_scale, output_scale=float(3.0 * sigma / 127.0) if case["kind"] == "int8_int8" else 1.0)
    weights = pla.detect_and_pack(dense, case["h"] * case["w"])
    kernel = pla.SparseConvKernel(pla.SparseConvParam(weights, bias=bias, activation_param=_activation(case["act"]), **param), *PRECISIONS[case["kind"]], reference_quirks=False)
    kernel.PrepareForRun()
    return kernel


def _input(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    shape = (case["batch"], case["ic"], case["h"], case["w"])
    if case["path"] == "quantised":
        return torch.randn(shape, device="cuda", generator=g) * 0.6
    if case["kind"] in ("fp32", "fp16"):
        return (torch.rand(shape, device="cuda", generator=g) * 2.0 - 1.0).to(torch.float32 if case["kind"] == "fp32" else torch.float16)
    return torch.randint(-127, 128, shape, device="cuda", dtype=torch.int8, generator=g)


def _body_shapes():
    """(depthwise stride, pointwise input channels, output channels, output side) of the thirteen blocks."""
    return [(s,) + t for s, t in zip(workloads.MOBILENET_V1_DEPTHWISE_STRIDES, workloads.MOBILENET_V1_POINTWISE)]


def _depthwise(channels, stride, seed):
    rng = np.random.RandomState(seed % 2**32)
    filt = rng.randint(-127, 128, size=(channels, 1, 3, 3)).astype(np.int8)
    weight_scale = rng.uniform(0.001, 0.02, size=channels).astype(np.float32)
    bias = (rng.standard_normal(channels) * 0.1).astype(np.float32)
    output_scale = 3.0 * 3.0 * 73.3 * 40.0 * float(weight_scale.mean()) * 0.01 / 127.0
    kernel = pla.DepthwiseConv(pla.ConvParam(filt, bias, strides=(stride, stride), paddings=(1, 1, 1, 1), activation_param=pla.ActivationParam("relu"), input_scale=0.01,
                                             weight_scale=weight_scale, output_scale=output_scale), out_precision="int8")
    kernel.PrepareForRun()
    return kernel


def _prepare_body(case, seed):
    """Layers, and one output buffer for each launch, as a program holds them that runs a network again and again."""
    batch = case["batch"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    blocks = _body_shapes()
    dws = [_depthwise(ic, stride, seed * 100 + i) for i, (stride, ic, _, _) in enumerate(blocks)]
    convs = [_conv({"kind": "int8_int8", "ic": ic, "oc": oc, "h": hw, "w": hw, "sparsity": case["sparsity"], "pairs": False, "act": "relu"}, seed * 100 + 50 + i)
             for i, (_, ic, oc, hw) in enumerate(blocks)]
    _, first_channels, _, first_side = blocks[0]
    x = torch.randint(-127, 128, (batch, first_channels, first_side, first_side), device="cuda", dtype=torch.int8, generator=g)
    steps = [(dws[0], None, torch.empty_like(x))]
    for i, (_, _, oc, hw) in enumerate(blocks):
        if i + 1 < len(blocks):
            side = blocks[i + 1][3]
            behind = torch.empty((batch, oc, side, side), device="cuda", dtype=torch.int8)
            if capi.lib().pl_sparse_conv_dwconv3x3_pays(convs[i]._handle, dws[i + 1]._handle, batch, hw, hw):
                steps.append((convs[i], dws[i + 1], behind))
                continue
        steps.append((convs[i], None, torch.empty((batch, oc, hw, hw), device="cuda", dtype=torch.int8)))
        if i + 1 < len(blocks):
            steps.append((dws[i + 1], None, behind))
    return {"path": "body", "x": x, "steps": steps}


def prepare(case, seed):
    if case["path"] == "body":
        return _prepare_body(case, seed)
    state = {"path": case["path"], "x": _input(case, seed), "kernel": _conv(case, seed)}
    if case["path"] == "quantised":
        state["q"] = torch.empty(state["x"].shape, device="cuda", dtype=torch.int8)
        state["calib"] = pla.CalibComputeFp32ToInt8(pla.CalibParam(state["x"], state["q"], 0.01))
        state["calib"].PrepareForRun()
    return state


def run(state):
    if state["path"] == "layer":
        return state["kernel"].Run(state["x"])
    if state["path"] == "quantised":
        state["calib"].Run(torch.cuda.current_stream().cuda_stream)
        return state["kernel"].Run(state["q"])
    x = state["x"]
    for first, behind, out in state["steps"]:
        if behind is None:
            x = first.Run(x, out)
        else:
            x = depthwise.run_conv_dw(first, behind, x, out)
    return x


def _layer_work(kind, batch, ic, oc, positions, sparsity):
    nonzeros = (1.0 - sparsity) * oc * ic
    weight_bytes = nonzeros * (IN_BYTES[kind] + 4) + 12.0 * oc
    return batch * positions * (ic * IN_BYTES[kind] + oc * OUT_BYTES[kind]) + weight_bytes, 2.0 * nonzeros * batch * positions


def work(case):
    if case["path"] == "body":
        total_bytes, flops = 0.0, 0.0
        batch = case["batch"]
        for stride, ic, oc, hw in _body_shapes():
            b, f = _layer_work("int8_int8", batch, ic, oc, hw * hw, case["sparsity"])
            total_bytes += b + batch * ic * hw * hw * (stride * stride + 1.0) + 17.0 * ic
            flops += f + 18.0 * batch * ic * hw * hw
        return {"bytes": total_bytes, "flops": flops}
    total_bytes, flops = _layer_work(case["kind"], case["batch"], case["ic"], case["oc"], case["h"] * case["w"], case["sparsity"])
    if case["path"] == "quantised":
        total_bytes += 5.0 * case["batch"] * case["ic"] * case["h"] * case["w"]
    return {"bytes": total_bytes, "flops": flops}


def tolerance(case):
    if case["path"] == "body":
        return "exact"
    # Against the same sums in 64 bits, over the listed layers and drawn ones: fp32 at most 3.2e-7 / 2.9e-6 (1024
    # channels), fp16, whose kernel accumulates in half precision, at most 2.3e-3 / 1.7e-2 (1568 channels).
    if case["kind"] == "fp32":
        return {"rel": 1.3e-6, "max": 1.2e-5}
    if case["kind"] == "fp16":
        return {"rel": 1e-2, "max": 7e-2}
    return "exact"
