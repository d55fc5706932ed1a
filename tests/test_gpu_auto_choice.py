"""The algorithm an automatic int8 handle picks must not lose much against the best forced one: the nine
distinct pointwise shapes of MobileNetV1-1.0 (int8 -> int8, relu, 90 % zeros) at 1, 4, 16 and 64 images per
launch, every algorithm the shape allows timed in the same process on the same buffers
(helpers.algo_times: parity-checked handles, interleaved runs, best of three).  A cell fails when the
automatic handle is more than 15 % (plus 0.3 us of timer resolution on these 4 to 17 us launches) slower than
the best forced algorithm."""
import numpy as np
import pytest

from helpers import algo_times, pla, workloads

pytestmark = pytest.mark.gpu

SHAPES = [(32, 64, 112), (64, 128, 56), (128, 128, 56), (128, 256, 28), (256, 256, 28), (256, 512, 14), (512, 512, 14), (512, 1024, 7), (1024, 1024, 7)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "%dx%d_%d" % s)
def test_auto_is_within_15_percent_of_the_best_forced_algorithm(shape):
    print("auto choice", shape, flush=True)
    index = workloads.MOBILENET_V1_POINTWISE.index(shape)
    slow = []
    for batch in (1, 4, 16, 64):
        case = workloads.config5_layer(index, batch=batch)
        times, picked = algo_times(case, warm=100, steps=400)
        best_name, best = min(((k, v) for k, v in times.items() if k != "auto"), key=lambda kv: kv[1])
        if times["auto"] > 1.15 * best + 0.3:
            # once more before failing: a burst on the box can land on one handle's runs
            times, picked = algo_times(case, warm=200, steps=800, repeats=5)
            best_name, best = min(((k, v) for k, v in times.items() if k != "auto"), key=lambda kv: kv[1])
            if times["auto"] > 1.15 * best + 0.3:
                slow.append("batch %d: auto (%s) %.2f us, %s %.2f us" % (batch, picked, times["auto"], best_name, best))
    assert not slow, "; ".join(slow)


# (batch, ic, oc, side, output): wide layers over several rounds of the workgroups that the device holds at once
WIDE_LAYERS = [(64, 2048, 2048, 14, "fp32"), (64, 2048, 2048, 14, "int8"), (24, 2048, 1024, 28, "fp32")]


@pytest.mark.parametrize("layer", WIDE_LAYERS, ids=lambda l: "%dx%dx%d_%d_%s" % l)
def test_auto_is_within_15_percent_on_wide_layers(layer):
    check_layer(*layer)


# calls at the borders of the rule for the kernel that takes the channels chunk by chunk: more than 512 channels over many
# positions, few of them through the row walk, small maps with 256 channels, channel blocks without weights
BORDERS = [(64, 520, 96, 56, "fp32"), (32, 520, 2048, 20, "fp32"), (128, 1280, 512, 20, "fp32"), (64, 1536, 2048, 17, "fp32"), (128, 1472, 812, 12, "int8"), (2, 96, 128, 10, "int8"),
           (32, 256, 256, 10, "fp32"), (2, 768, 256, 8, "fp32"), (128, 192, 384, 13, "int8"), (16, 2048, 2048, 14, "fp32"), (64, 192, 384, 17, "fp32"), (16, 600, 600, 12, "fp32"),
           (65, 492, 101, 32, "fp32"), (68, 360, 327, 28, "fp32"), (181, 581, 267, 24, "fp32"), (24, 512, 384, 28, "fp32"), (67, 1024, 1920, 7, "int8")]


@pytest.mark.parametrize("layer", BORDERS, ids=lambda l: "%dx%dx%d_%d_%s" % l)
def test_auto_is_within_15_percent_at_the_borders_of_the_chunk_rule(layer):
    check_layer(*layer)


@pytest.mark.parametrize("layer", [(64, 1024, 1024, 20, "fp32"), (16, 2048, 2048, 14, "fp32"), (128, 2048, 2048, 8, "fp32")], ids=lambda l: "%dx%dx%d_%d_%s" % l)
def test_auto_is_within_15_percent_with_empty_blocks(layer):
    check_layer(*layer, sparsity=0.95, blocked=True)


def check_layer(batch, ic, oc, side, out, sparsity=0.85, blocked=False):
    print("auto choice", batch, ic, oc, side, out, sparsity, blocked, flush=True)
    case = workloads.make_int8("%dx%dx%d_%d" % (batch, ic, oc, side), batch, ic, oc, side, side, sparsity, False, pla.ActivationParam("leaky_relu", Leaky_relu_alpha=0.1), out_int8=out == "int8", seed=ic + oc,
                               output_scale=0.2 * (ic / 64.0)**0.5 if out == "int8" else 1.0)
    if blocked:  # whole 32 x 32 blocks of zeros
        keep = np.random.RandomState(ic).random_sample((oc // 32, ic // 32)) >= sparsity
        case.dense = (workloads._int8_nonzero(np.random.RandomState(oc), (oc, ic)) * np.kron(keep, np.ones((32, 32), dtype=bool))).astype(np.int8)
    times, picked = algo_times(case, warm=30, steps=100, chunk_positions=(64, 128, 256, "split"))
    best_name, best = min(((k, v) for k, v in times.items() if k != "auto"), key=lambda kv: kv[1])
    if times["auto"] > 1.15 * best + 0.3:
        times, picked = algo_times(case, warm=60, steps=200, repeats=5, chunk_positions=(64, 128, 256, "split"))
        best_name, best = min(((k, v) for k, v in times.items() if k != "auto"), key=lambda kv: kv[1])
    assert times["auto"] <= 1.15 * best + 0.3, "auto (%s) %.2f us, %s %.2f us" % (picked, times["auto"], best_name, best)
