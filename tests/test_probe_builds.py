"""The measurement builds go through a wave's units as the product's build of the same launch does: one, two, the first two
requested together, or any number in a loop."""
import os
import re

import numpy as np
import pytest

import mixed_gemv_amd as mg
from mixed_gemv_amd import build as lib_build
from helpers import SCALE_AND_ZEROS, DeviceProblem, Problem

FORMS = (mg.UNIT_FORM_LOOP, mg.UNIT_FORM_ONE, mg.UNIT_FORM_TWO, mg.UNIT_FORM_TWO_AHEAD)


def test_every_way_through_the_units_has_its_measurement_builds():
    asm = os.path.join(lib_build.OBJ_DIR, "probes-hip-amdgcn-amd-amdhsa-gfx950.s")
    if not os.path.exists(asm):
        pytest.skip("no device assembly: built elsewhere")
    builds = set(re.findall(r"^ +\.symbol: +\S*gemv_dpp_kernelILi4ELi3ELi1ELi1ELb0ELi0ELi(\d)ELi(\d)ELb0E\S*\.kd$", open(asm).read(), re.M))
    assert builds == {(str(probe), str(form)) for probe in (1, 2, 3) for form in FORMS}


@pytest.mark.gpu
@pytest.mark.parametrize("n_out, k, form", [(1024, 2048, mg.UNIT_FORM_ONE), (4096, 4096, mg.UNIT_FORM_TWO),
                                            (4096, 4608, mg.UNIT_FORM_TWO_AHEAD),      # three units a wave
                                            (1024, 10240, mg.UNIT_FORM_TWO_AHEAD),     # five
                                            (17600, 10240, mg.UNIT_FORM_LOOP),         # waves that share the SIMDs
                                            (28672, 8192, mg.UNIT_FORM_LOOP)])         # walks of tiles
def test_measurement_builds_of_every_form(gpu, n_out, k, form):
    import torch
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    if cus != 256:
        pytest.skip("the launches are chosen for a device of 256 compute units")
    assert mg.probe_unit_form(n_out, 1, k, 4, 128) == form
    plan = mg.query_launch(n_out, 1, k, 4, 128, num_compute_units=cus)
    prob = Problem("probe_form", n_out, k, 4, SCALE_AND_ZEROS, 128, x_dist="normal")
    dev = DeviceProblem(prob, gpu)
    want = dev.run().copy().view(np.uint16)
    waves = -(-plan["workgroups"] // 8) * 8 * plan["threads"] // 64
    for kind in (mg.PROBE_TIMELINE, mg.PROBE_TIMELINE_WAITS):
        trace = torch.zeros((waves, mg.PROBE_TIMELINE_WORDS), dtype=torch.int64, device=gpu)
        dev.y.fill_(0x7e00)
        mg.probe_gemv(kind, trace, dev.w, dev.x, dev.scale, dev.zero, dev.y, n_out, k, 128)
        torch.cuda.synchronize()
        assert np.array_equal(dev.y.cpu().numpy().view(np.uint16), want)
        t = trace.cpu().numpy()
        t = t[t[:, 0] > 0]
        assert np.all(np.diff(t[:, :5], axis=1) >= 0)
        assert t[:, 11].sum() == n_out // 16 * -(-k // 512)                # every unit, once
        assert np.all(t[:, 5:8].sum(axis=1) <= t[:, 3] - t[:, 1])
    for kind in (mg.PROBE_LOADS_ONLY, mg.PROBE_COMPUTE_ONLY):
        dev.y.fill_(0x7e00)
        mg.probe_gemv(kind, None, dev.w, dev.x, dev.scale, dev.zero, dev.y, n_out, k, 128)
        torch.cuda.synchronize()
        assert not np.any(dev.y.cpu().numpy().view(np.uint16) == 0x7e00)
