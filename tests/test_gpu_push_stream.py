"""Level 0's pass beside the finer levels' on a stream of its own, which it takes
between 64 and 256 MB of level 0's two buffers: several steps enqueued at once
equal steps with reads of every level between them, bit for bit, on either side
of both bounds."""
import numpy as np
import pytest

from lambrex_amd import lbx, workloads
from test_gpu_multilevel import gpu_levels, make_gpu, masks_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edge", [62, 68, 100, 106])  # 57, 75, 240 and 286 MB
def test_steps_at_once_equal_steps_with_reads(ctx, edge):
    dims = (edge,) * 3
    levels = [workloads.chop(dims, 64), [((16, 16, 16), (47, 79, 63)), ((48, 16, 16), (79, 79, 63))],
              [((64, 64, 64), (95, 111, 95))]]
    masks = masks_for("fine", levels)
    rho, u = workloads.random_state(dims, 3, 1e-2, 0.02)
    out = []
    for chunks in ((6,), (1,) * 6):
        sim = make_gpu(ctx, dims, levels, masks, 0.8, rho, u)
        for n in chunks:
            sim.iterate(n)
            got = gpu_levels(sim, len(levels))
        sim.close()
        out.append(got)
    for a, b in zip(*out):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
