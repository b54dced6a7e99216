"""The Python device entry points' argument handling (csrc/py_calls.cpp): what they take, and what they refuse."""
import os
import subprocess
import sys

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


WITHOUT_TORCH = """
import sys
sys.modules["torch"] = None      # import torch raises ImportError from here on
import numpy as np
import mixed_gemv_amd as mg
from mixed_gemv_amd import build

def status(call):
    try:
        call()
    except mg.MixedGemvError as e:
        return e.status
    return 0

p = 0x1000
number = np.int64
assert status(lambda: mg.device_gemv(p, p, p, p, None, p, 1, number(18), 1, 512, 128, stream=0)) == 3
assert status(lambda: mg.device_gemv(p, p, p, p, None, p, 0, 16, 1, 512, 128, stream=0, element="bf16")) == 8
assert status(lambda: mg.device_gemv(p, p, p, p, None, p, -2, 16, 1, 512, 128, stream=0, batch_strides=(1, 0, 0, 0, 0))) == 8
assert status(lambda: mg.device_gemv(None, p, p, p, None, p, 1, 16, 1, 512, 128, stream=0)) == 1
for element in (None, "f16", "bf16"):
    assert status(lambda: mg.device_gemv_routed(p, p, p, p, None, p, None, 4, 2, 16, 1, 512, 128, [0] * 5, stream=0, element=element)) == 1
    assert status(lambda: mg.dequantize(p, p, p, p, 16, 511, 128, stream=0, element=element)) == 4
for call in (lambda: mg.device_gemv("w", p, p, p, None, p, 1, 16, 1, 512, 128, stream=0),
             lambda: mg.device_gemv(p, p, p, p, None, p, 1, 16, 1, 512, 128, stream=0, batch_strides=(1, 2)),
             lambda: mg.device_gemv(p, p, p, p, None, p, 1, 16, 1, 512, 128)):
    try:
        call()
    except (TypeError, ValueError, ImportError):   # no address; no five strides; no current stream to ask for
        continue
    raise AssertionError("accepted")
build.PY_CALLS_PATH = sys.argv[1]
open(sys.argv[1], "w").close()
assert build.build_py_calls() is None
import os
assert not os.path.exists(sys.argv[1])
print("ok")
"""


def test_addresses_and_the_build_work_without_pytorch(tmp_path):
    repo = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", WITHOUT_TORCH, str(tmp_path / "py_calls.so")], cwd=repo,
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


@pytest.mark.parametrize("element,suffix", [(None, ""), ("f16", ""), ("bf16", "_bf16")])
def test_the_ctypes_calls_hand_every_argument_to_its_place(monkeypatch, element, suffix):
    from mixed_gemv_amd import api
    seen = []

    class Recorder:
        def __getattr__(self, name):
            return lambda *a: seen.append((name, [getattr(v, "value", v) for v in a])) or 0

    monkeypatch.setattr(api, "_lib", type("Lib", (), {"lib": staticmethod(Recorder)}))
    monkeypatch.setattr(api, "_calls", api._CtypesCalls)
    mg.device_gemv(1, 2, 3, None, 5, 6, 7, 8, np.int64(9), 10, 11, 12, 13, stream=14, element=element)
    mg.device_gemv(1, 2, 3, 4, None, 6, 7, 8, 9, 10.0, 11, 12, 13, stream=14, batch_strides=[15, 16, 17, 18, 19], element=element)
    mg.device_gemv_routed(1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, (14, 15, 16, 17, 18), 19, 20, stream=21, element=element)
    mg.dequantize(1, 2, 3, 4, 5, 6, 7, 8, 9, stream=10, element=element)
    assert seen == [
        ("mgemv_gemv_batched" + suffix, [1, 2, 3, None, 5, 6, 7, 8, 9, 10, 11, 12, 13, 0, 0, 0, 0, 0, 14]),
        ("mgemv_gemv_batched" + suffix, [1, 2, 3, 4, None, 6, 7, 8, 9, 10, 11, 12, 13, 15, 16, 17, 18, 19, 14]),
        ("mgemv_gemv_routed" + suffix, [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 19, 20, 14, 15, 16, 17, 18, 21]),
        ("mgemv_dequantize" + suffix, [1, 2, 3, 4, 5, 6, 7, 8, 9, 10])]
