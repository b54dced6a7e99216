"""The Python device entry points' argument handling (csrc/py_calls.cpp): what they take, and what they refuse."""
import numpy as np
import pytest
import torch

import mixed_gemv_amd as mg
from helpers import SCALE_AND_ZEROS, DeviceProblem, Problem
from mixed_gemv_amd import MixedGemvError


def test_addresses_that_are_no_gpu_tensor():
    cpu = torch.zeros(64, dtype=torch.half)
    with pytest.raises(ValueError, match="GPU tensors"):
        mg.device_gemv(cpu, cpu, cpu, cpu, None, cpu, 1, 16, 1, 512, 128, stream=0)
    with pytest.raises(TypeError, match="device address"):
        mg.dequantize(np.zeros(4), None, None, None, 16, 512, 128, stream=0)
    with pytest.raises(ValueError, match="element must be"):
        mg.device_gemv(0x1000, 0x1000, 0x1000, 0x1000, None, 0x1000, 1, 16, 1, 512, 128, stream=0, element="f32")
    with pytest.raises(ValueError, match="five"):
        mg.device_gemv(0x1000, 0x1000, 0x1000, 0x1000, None, 0x1000, 2, 16, 1, 512, 128, stream=0, batch_strides=(1, 2))
    with pytest.raises(TypeError):
        mg.device_gemv(0x1000, 0x1000, 0x1000, 0x1000, None, 0x1000, 1, "16", None, 512, 128, stream=0)


@pytest.mark.parametrize("number", [int, np.int64, np.int32, float])
def test_numbers_of_any_kind_reach_the_argument_checks(number):
    def status(call):
        with pytest.raises(MixedGemvError) as ei:
            call()
        return ei.value.status

    p = 0x1000
    assert status(lambda: mg.device_gemv(p, p, p, p, None, p, 1, number(18), 1, number(512), 128, stream=0)) == 3
    assert status(lambda: mg.device_gemv(p, p, p, p, None, p, number(0), 16, 1, 512, 128, stream=0)) == 8
    assert status(lambda: mg.device_gemv(None, p, p, p, None, p, 1, 16, 1, 512, number(128), stream=0)) == 1
    assert status(lambda: mg.device_gemv_routed(p, p, p, p, None, p, None, 4, 2, 16, 1, 512, 128, [number(0)] * 5, stream=0)) == 1
    assert status(lambda: mg.dequantize(p, p, p, p, 16, number(511), 128, stream=0)) == 4


@pytest.mark.gpu
def test_tensors_addresses_streams_and_element_types_give_the_same_bits(gpu):
    prob = Problem("py_calls", 80, 1024, 4, SCALE_AND_ZEROS, 128, bias=True)
    d = DeviceProblem(prob, gpu)
    want = d.run()
    sizes = (1, prob.n_out, 1, prob.k, 128, mg.WeightOnlyQuantOp.FINEGRAINED_SCALE_AND_ZEROS, 4)
    side = torch.cuda.Stream()
    for stream in (None, side, side.cuda_stream, 0):
        for addresses in (False, True):
            ops = [d.w, d.x, d.scale, d.zero, d.bias, d.y]
            d.y.zero_()
            torch.cuda.synchronize()
            mg.device_gemv(*[o.data_ptr() for o in ops] if addresses else ops, *sizes, stream=stream)
            torch.cuda.synchronize()
            assert np.array_equal(d.y.cpu().numpy().view(np.uint16).reshape(-1), np.asarray(want).view(np.uint16).reshape(-1))
    with torch.cuda.stream(side):   # the current stream is the one that is taken
        d.y.zero_()
        mg.device_gemv(d.w, d.x, d.scale, d.zero, d.bias, d.y, *sizes)
        side.synchronize()
        assert np.array_equal(d.y.cpu().numpy().view(np.uint16).reshape(-1), np.asarray(want).view(np.uint16).reshape(-1))
    strided = torch.zeros((2 * prob.n_out,), dtype=torch.half, device=gpu)[::2]
    with pytest.raises(ValueError, match="contiguous"):
        mg.device_gemv(d.w, d.x, d.scale, d.zero, d.bias, strided, *sizes)
