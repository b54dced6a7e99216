"""What the tuner measures candidates and entries against: the plan a launch takes by itself, parts of tiles included, and not the rules
behind the measured ranges.  The times come from the plan in force, so no GPU is needed."""
import types

import pytest
import torch

import mixed_gemv_amd as mg
from mixed_gemv_amd import autotune

SHAPES = [(1024, 16384, 1, "f16"),     # a single row on few tiles
          (2048, 11008, 4, "f16"),     # several rows on few tiles
          (5004, 4608, 3, "bf16")]     # tiles left over from a walk of one
ENTRY = dict(kernel=mg.KERNEL_VALU, split_k=4, tiles_per_wg=1)


def plan(n_out, k, rows, element):
    args = dict(weight_bits=4, group_size=128, element=element, num_compute_units=256)
    return mg.query_launch(n_out, rows, k, **args), mg.plan_coverage(n_out, rows, k, **args)


@pytest.fixture
def timed(monkeypatch):
    """Times by plan: what the launch takes by itself 5 us, everything else 7."""
    built_in = {}

    class Timed:
        def __init__(self, n_out, k, bits, qop, group, rows, bias, device, seed, cold_bytes, element):
            self.shape = (n_out, k, rows, element)

        def time_us(self, launches):
            return 5.0 if plan(*self.shape) == built_in[self.shape] else 7.0

    autotune.clear()
    for shape in SHAPES:
        built_in[shape] = plan(*shape)
    monkeypatch.setattr(autotune, "_Problem", Timed)
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda d: types.SimpleNamespace(multi_processor_count=256))
    monkeypatch.setattr(torch.cuda, "device", lambda d: __import__("contextlib").nullcontext())
    yield built_in
    autotune.clear()


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_nothing_is_installed_over_a_faster_built_in_plan(timed, shape):
    n_out, k, rows, element = shape
    mg.set_tuned_plan(n_out, k, 4, 128, rows, **ENTRY, element=element)     # a poor entry of an earlier run
    res = autotune.tune(n_out, k, 4, 3, 128, m_batch=rows, element=element, launches=1, rounds=1)
    assert res["builtin_geometry"] == timed[shape][0] and res["builtin_us"] == 5.0
    assert res["entry"] is None and all(us == 7.0 for us, _ in res["measurements"][1:]) and len(res["measurements"]) > 4
    assert plan(*shape) == timed[shape] and mg.tuned_plan_count() == 0


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_an_entry_is_confirmed_against_the_built_in_plan_and_stays(timed, shape):
    n_out, k, rows, element = shape
    entry = dict(n_out=n_out, k=k, weight_bits=4, group_size=128, m_batch=rows, element=element, **ENTRY)
    mg.set_tuned_plan(**entry)
    tuned = plan(*shape)
    assert tuned != timed[shape]
    assert autotune.reconfirm(entry, launches=1, rounds=1) == round(100 * (5 / 7 - 1), 2)
    assert plan(*shape) == tuned and mg.tuned_plan_count() == 1


def test_a_shipped_entry_is_confirmed_against_the_rules(timed, monkeypatch):
    shape = (28672, 8192, 1, "f16")
    timed[shape] = plan(*shape)
    entry = dict(n_out=28672, k=8192, weight_bits=4, group_size=128, m_batch=1, kernel=mg.KERNEL_VALU, split_k=8, tiles_per_wg=1,
                 max_workgroups=256)
    assert autotune.reconfirm(entry, launches=1, rounds=1) == 40.0
