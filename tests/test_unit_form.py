"""Which build of the VALU kernel a launch takes (unit_form in csrc/kernel_common.h): by the length of its waves, and for waves
of three and more units by whether all problems of the launch together leave each wave a SIMD to itself."""
import numpy as np
import pytest

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem

LOOP, TWO, AHEAD, ONE = mg.UNIT_FORM_LOOP, mg.UNIT_FORM_TWO, mg.UNIT_FORM_TWO_AHEAD, mg.UNIT_FORM_ONE


@pytest.mark.parametrize("n_out, rows, k, bits, element, batch, cus, form", [
    (4096, 1, 4096, 4, "f16", 1, 256, TWO), (4096, 1, 4096, 4, "f16", 8, 256, TWO),
    (1024, 1, 2048, 4, "f16", 1, 256, ONE), (1024, 1, 2048, 4, "f16", 64, 256, ONE),
    (4096, 1, 4096, 8, "f16", 1, 256, AHEAD), (4096, 1, 4096, 8, "f16", 3, 256, LOOP),   # 256 x 4 waves of four units
    (2048, 1, 11008, 4, "f16", 2, 256, AHEAD), (2048, 1, 11008, 4, "f16", 3, 256, LOOP),  # 128 x 4
    (2048, 2, 11008, 4, "bf16", 2, 256, AHEAD), (2048, 2, 11008, 4, "bf16", 3, 256, LOOP),
    (2048, 1, 11008, 4, "f16", 1, 64, AHEAD), (2048, 1, 11008, 4, "f16", 2, 64, LOOP),      # 64 pairs of tiles x 2 x 2
    (28672, 1, 8192, 4, "f16", 1, 256, LOOP),     # walks
    (8192, 8, 8192, 4, "f16", 1, 256, LOOP)])     # matrix cores
def test_build_of_a_launch(n_out, rows, k, bits, element, batch, cus, form):
    assert mg.probe_unit_form(n_out, rows, k, bits, 128, element, batch, cus) == form


def test_single_stage_launches_take_the_loop():
    try:
        mg.set_prefetch_stages(1)
        assert [mg.probe_unit_form(n, 1, k) for n, k in ((4096, 4096), (1024, 2048), (2048, 11008))] == [LOOP] * 3
    finally:
        mg.set_prefetch_stages(0)


@pytest.mark.gpu
@pytest.mark.parametrize("element", ["f16", "bf16"])
@pytest.mark.parametrize("bits, qop, group, ksteps, rows", [(4, SCALE_AND_ZEROS, 128, 17, 1), (4, SCALE_ONLY, 96, 18, 1),
                                                            (8, PER_COLUMN, 0, 19, 1), (8, SCALE_AND_ZEROS, 64, 17, 3)])
def test_batched_launches_have_the_bits_of_single_ones_in_either_build(gpu, bits, qop, group, ksteps, rows, element):
    import torch
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    step = 512 if bits == 4 else 256
    n_out, most = 1032, 6                      # 65 tiles of four waves: three problems are 780 waves, six 1560
    k = (ksteps * step - step // 2) // (8 if qop == PER_COLUMN else group) * (8 if qop == PER_COLUMN else group)
    probs = [Problem(f"form{b}", n_out, k, bits, qop, group, m_batch=rows, bias=True, element=element) for b in range(most)]
    devs = [DeviceProblem(p, gpu) for p in probs]
    cat = lambda name: None if getattr(devs[0], name) is None else torch.stack([getattr(d, name) for d in devs])  # noqa: E731
    w, x, scale, zero, bias = (cat(n) for n in ("w", "x", "scale", "zero", "bias"))
    strides = (w[0].numel(), rows * k, scale[0].numel(), n_out, rows * n_out)
    want = np.stack([d.run().copy().view(np.uint16).reshape(rows, n_out) for d in devs])
    forms = set()
    for batch in (3, most):
        forms.add(mg.probe_unit_form(n_out, rows, k, bits, probs[0].group_size, element, batch, cus))
        y = torch.full((batch, rows, n_out), 0x7E00, dtype=torch.int16, device=gpu)
        mg.device_gemv(w, x, scale, zero, bias, y, batch, n_out, rows, k, probs[0].group_size, qop, bits, batch_strides=strides,
                       element=element)
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy().view(np.uint16), want[:batch]), batch
    assert cus != 256 or forms == {AHEAD, LOOP}
