"""What the Python classes' Run looks up once and what it passes by: a second PrepareForRun with other layers, a stream
that the caller names, a current device that is not the tensor's."""
import importlib

import numpy as np
import pytest

from helpers import capi, make_kernel, pla, run_oracle, workloads
from test_gpu_conv_dw_fused import make_pair

pytestmark = pytest.mark.gpu
depthwise = importlib.import_module("paddle-lite_amd.depthwise_conv")
AP = pla.ActivationParam


def _layer(ic, oc, out_int8):
    return workloads.make_int8("run", 2, ic, oc, 5, 6, 0.8, False, AP("relu"), out_int8=out_int8, seed=ic, output_scale=0.2)


def _host(t):
    import torch

    torch.cuda.synchronize()
    return t.cpu().numpy()


def test_second_prepare_with_other_channels():
    import torch

    first, second = _layer(70, 24, False), _layer(200, 56, False)
    kernel, _ = make_kernel(first)
    assert np.array_equal(_host(kernel.Run(torch.from_numpy(first.x).cuda())), run_oracle(first))
    kernel.param = make_kernel(second)[0].param
    kernel.PrepareForRun()
    x = torch.from_numpy(second.x).cuda()
    assert np.array_equal(_host(kernel.Run(x)), run_oracle(second))
    with pytest.raises(ValueError):
        kernel.Run(torch.from_numpy(first.x).cuda())
    # the depthwise class likewise: channels, stride and padding
    _, _, dw, _ = make_pair(1, 128, 128, 1, "relu", "relu", 3)
    _, _, other, _ = make_pair(1, 128, 256, 2, "relu", "relu", 4)
    y = torch.randint(-127, 128, (2, 256, 9, 8), dtype=torch.int8, device="cuda")
    dw.Run(y[:, :128].contiguous())
    dw.param = other.param
    dw.PrepareForRun()
    got, want = dw.Run(y), other.Run(y)
    assert tuple(got.shape) == (2, 256, 5, 4) and torch.equal(got, want)


def test_a_stream_that_the_caller_names():
    """Behind work on that stream, with nothing of it on the current one: the result is there once that stream is done."""
    import torch

    case, conv, dw, _ = make_pair(2, 128, 128, 2, "relu", "relu", 5)
    x = torch.from_numpy(case.x).cuda()
    mid = conv.Run(x)
    out = dw.Run(mid)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    late = torch.zeros_like(x)
    late_mid, late_out, fused = torch.zeros_like(mid), torch.zeros_like(out), torch.zeros_like(out)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        busy = torch.randn(2048, 2048, device="cuda")
        for _ in range(4):
            busy = busy @ busy * 1e-3
        late.copy_(x)
    conv.Run(late, late_mid, stream=side.cuda_stream)
    dw.Run(late_mid, late_out, stream=side.cuda_stream)
    depthwise.run_conv_dw(conv, dw, late, fused, stream=side.cuda_stream)
    side.synchronize()
    assert torch.equal(late_mid, mid) and torch.equal(late_out, out) and torch.equal(fused, out)


def test_the_current_device_is_not_the_tensors(monkeypatch):
    """The depthwise calls enter the tensor's device where another one is current; here the current one is only said to be
    another, so that the calls must still give their results."""
    import torch

    case, conv, dw, _ = make_pair(2, 128, 128, 1, "relu", "relu", 6)
    x = torch.from_numpy(case.x).cuda()
    mid = conv.Run(x)
    out = dw.Run(mid)
    entered = []
    real = torch.cuda.device

    class Entering(real):
        def __init__(self, device):
            entered.append(torch.device(device))
            super().__init__(device)

    monkeypatch.setattr(torch.cuda, "current_device", lambda: x.device.index + 1)
    monkeypatch.setattr(torch.cuda, "device", Entering)
    assert torch.equal(dw.Run(mid), out) and entered == [x.device]
    assert torch.equal(depthwise.run_conv_dw(conv, dw, x), out) and entered == [x.device] * 2
