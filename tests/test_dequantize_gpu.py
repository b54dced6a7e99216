"""The dequantise kernel at the edges of its units, with tables and outputs at the least alignment the boundary takes."""
import numpy as np
import pytest
import torch

import mixed_gemv_amd as mg
from helpers import PER_COLUMN, SCALE_AND_ZEROS, SCALE_ONLY, DeviceProblem, Problem

pytestmark = pytest.mark.gpu


def shifted(t, elements, device):
    """The same values `elements` 16-bit elements past an aligned address."""
    flat = torch.zeros((t.numel() + elements,), dtype=t.dtype, device=device)
    flat[elements:] = t.reshape(-1)
    return flat[elements:]


@pytest.mark.parametrize("element", ["f16", "bf16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("n_out,k,op,group", [
    (4, 8, PER_COLUMN, 8),                  # one piece of one row
    (20, 520, PER_COLUMN, 520),             # one piece past a k step, a quarter of a second tile
    (36, 1088, SCALE_AND_ZEROS, 64),        # group and k step end apart
    (100, 768, SCALE_ONLY, 96),
    (64, 2048, SCALE_AND_ZEROS, 128),
])
def test_edges_and_least_alignment(gpu, n_out, k, op, group, bits, element):
    prob = Problem("dequantize", n_out, k, bits, op, group, element=element)
    d = DeviceProblem(prob, gpu)
    want = prob.oracle_dequant().view(np.uint16)
    for off in (0, 1, 3):   # tables: 2-byte aligned; outputs: 4-byte aligned
        scale = shifted(d.scale, off, gpu)
        zero = shifted(d.zero, off, gpu) if d.zero is not None else None
        room = torch.full((n_out * k + 16,), 0x7e01, dtype=torch.int16, device=gpu)
        out = room[2 * off:2 * off + n_out * k]
        mg.dequantize(d.w, scale, zero, out, n_out, k, group, op, bits, element=element)
        torch.cuda.synchronize()
        got = room.cpu().numpy().view(np.uint16)
        assert np.array_equal(got[2 * off:2 * off + n_out * k].reshape(n_out, k), want)
        assert (got[:2 * off] == 0x7e01).all() and (got[2 * off + n_out * k:] == 0x7e01).all()
