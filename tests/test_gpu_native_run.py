"""The native part of the Python classes' Run (csrc/python_run.cc): it takes the common call, gives what the Python code
gives, and leaves every other call to that."""
import importlib

import numpy as np
import pytest

from helpers import capi, make_kernel, pla, workloads
from test_gpu_conv_dw_fused import make_pair

pytestmark = pytest.mark.gpu
depthwise = importlib.import_module("paddle-lite_amd.depthwise_conv")


def _layers():
    import torch

    case, conv, dw, _ = make_pair(3, 128, 128, 2, "relu", "relu", 8)
    x = torch.from_numpy(case.x).cuda()
    return conv, dw, x


def test_the_common_call_is_native(monkeypatch):
    import torch

    conv, dw, x = _layers()
    mid = conv.Run(x)
    out = dw.Run(mid)
    fused = depthwise.run_conv_dw(conv, dw, x)
    for layer in (conv, dw):
        monkeypatch.setattr(type(layer), "_run", lambda *a: pytest.fail("the Python code ran"))
    assert torch.equal(conv.Run(x), mid) and torch.equal(dw.Run(mid), out)
    for target, run in ((torch.zeros_like(mid), lambda t: conv.Run(x, t)), (torch.zeros_like(out), lambda t: dw.Run(mid, t)), (torch.zeros_like(fused), lambda t: depthwise.run_conv_dw(conv, dw, x, t))):
        want = run(None)
        assert want.dtype == target.dtype and want.device == target.device and not want.requires_grad
        assert run(target) is target and torch.equal(target, want)


@pytest.mark.parametrize("kind", ["fp32", "fp16", "int8_fp32"])
def test_types(kind):
    import torch

    if kind == "int8_fp32":
        case = workloads.make_int8("t", 2, 70, 24, 5, 6, 0.8, False, pla.ActivationParam("relu"), out_int8=False, seed=1)
    else:
        case = workloads.make_fp32("t", 2, 70, 24, 5, 6, 0.8, False, pla.ActivationParam("relu"), seed=1)
        if kind == "fp16":
            case.kind, case.x = capi.KIND_FP16, case.x.astype(np.float16)
    kernel, _ = make_kernel(case)
    x = torch.from_numpy(case.x).cuda()
    first, second = kernel.Run(x), kernel.Run(x)
    assert kernel._native is not None and first.dtype == second.dtype and torch.equal(first, second)
    # the stream that is current
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        third = kernel.Run(x)
    side.synchronize()
    assert torch.equal(first, third)


def test_other_calls_are_left_to_the_python_code():
    """Each refused as before, with the native function in place; nothing is written."""
    import torch

    conv, dw, x = _layers()
    mid = conv.Run(x)
    want = dw.Run(mid)
    conv.Run(x), dw.Run(mid)
    assert conv._native is not None and dw._native is not None
    for bad in (x.cpu(), x.float(), x[:, :64].contiguous(), x.transpose(2, 3), x[0], x.double()):
        with pytest.raises(ValueError):
            conv.Run(bad)
        with pytest.raises(ValueError):
            depthwise.run_conv_dw(conv, dw, bad)
    for bad in (mid.cpu(), mid.float(), mid[:, :64].contiguous(), mid.transpose(2, 3)):
        with pytest.raises(ValueError):
            dw.Run(bad)
    for layer, source, good in ((conv, x, mid), (dw, mid, want)):
        for bad in (torch.zeros_like(good)[:1], torch.zeros_like(good).float(), torch.zeros_like(good).cpu(), torch.zeros_like(good).transpose(2, 3)):
            with pytest.raises(ValueError):
                layer.Run(source, bad)
            assert not bad.any()
    # a subclass of tensor, and a stream given as something else than a number, still run
    class Sub(torch.Tensor):
        pass

    assert torch.equal(conv.Run(x.as_subclass(Sub)).as_subclass(torch.Tensor), mid)
    import ctypes as C

    assert torch.equal(conv.Run(x, None, C.c_void_p(torch.cuda.current_stream().cuda_stream)), mid)
    # an empty batch is no work
    assert tuple(conv.Run(x[:0]).shape) == (0,) + tuple(mid.shape[1:])
    # a handle that is gone
    conv._release()
    with pytest.raises(RuntimeError):
        conv.Run(x)
