"""Every increment of the quality-guided unwrapping on fields of random phase:
tests/golden/herraez_phase.npz holds the phases (float16) that the reference's
merge sort, replayed level by level, followed by a spanning tree on the sorted
positions, gave for these crops. Another spanning tree moves pixels by multiples
of 2 pi; rounding (of the storage: phases up to 256 to 0.125, of the fit: less)
stays below 0.2."""
import os

import numpy as np
import pytest

from cases import LAM, N0, NA

GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "herraez_phase.npz")
# one tile, two depths of edge ranges, ragged tiles, components in LDS and not
SIDES = [32, 34, 70, 128, 256]


def crops(C):
    """A specular over noise of its size, by integer arithmetic alone."""
    y, x = np.mgrid[0:C, 0:C].astype(np.int64)
    s = (x * 7919 + y * 104729 + x * y * 31 + C) * 2654435761 % (1 << 32)
    t = (s ^ (s >> 15)) * 2246822519 % (1 << 32)
    c = ((s >> 11) % 401 - 200) + 1j * ((t >> 13) % 401 - 200)
    c[0, 0] = 0
    c[3, 5] = 1200
    return c[None].astype(np.complex64)


def phases(m, ctx, C):
    import torch
    nx = C // 2
    g = m.geom_derive(8 * nx, nx, 4 * nx, 4 * nx, 4 * nx, NA, N0, LAM, nx * LAM / (NA * 8 * nx),
                      born=0, c_aber=1, deroul=2)
    pos = torch.empty((2,), dtype=torch.int32, device="cuda")
    f = torch.empty((1, C, C), dtype=torch.complex64, device="cuda")
    ctx.crop_to_field(g, torch.from_numpy(crops(C)).cuda(), None, pos, f)
    assert pos.tolist() == [5, 3]
    return f.imag.cpu().numpy()[0]


@pytest.mark.gpu
@pytest.mark.parametrize("C", SIDES)
def test_increments(gpu_ctx, C):
    import mtd_transmission_amd as m
    want = np.load(GOLDEN)["c%d" % C].astype(np.float64)
    print(C, flush=True)
    assert np.abs(phases(m, gpu_ctx, C) - want).max() < 0.2
    assert np.ptp(want) > 4 * np.pi  # there are increments to get wrong
