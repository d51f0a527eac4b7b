"""The whole-step pass over a refined level (k_fine_step) at the edges of its
tiles, against the CPU oracle: boxes of 2 cells, boxes wider than a tile in x
and y, boxes cut in z, boxes of different shapes (whose population strides
differ) in any order, a box that is its own neighbour through the periodic
faces, and the same on a level between level 0 and the finest.

FP64 is bitwise.  FP32-shifted storage is held to the FP64 oracle: a (sub)step
rounds a population about 40 times by 2^-24 of at most the largest one, 2 coarse
steps of 3 levels are 8 substeps, and the fills, sums and the growth of an error
from one substep to the next are given a factor of 4: 4 * 8 * 40 * 2^-24 = 8e-5
of the largest population.  A wrong source or plane is off by the state's
variation, 1e-2 of it."""
import numpy as np
import pytest

from lambrex_amd import lbx, workloads
from oracle import oracle as orc
from test_gpu_multilevel import gpu_levels, make_gpu, masks_for, run_oracle
from test_gpu_twolevel import assert_bitwise, fine_boxes_in

pytestmark = pytest.mark.gpu

TALL = ((4, 4, 0), (9, 9, 127))
WIDE = ((10, 4, 10), (23, 15, 29))

CASES = {  # coarse extents, boxes of each refined level
    "two_cells": ((8, 8, 8), [fine_boxes_in((4, 4, 4), (9, 9, 9), 2)]),
    "wide": ((40, 44, 6), [[((4, 2, 0), (75, 71, 11))]]),
    "tall": ((14, 10, 64), [[TALL, WIDE]]),
    "other_order": ((14, 10, 64), [[WIDE, TALL]]),
    "whole_domain": ((5, 20, 7), [[((0, 0, 0), (9, 39, 13))]]),
    "slabs": ((36, 4, 4), [fine_boxes_in((0, 2, 2), (71, 5, 5), 40)]),
    "three": ((20, 20, 24), [[((4, 4, 4), (37, 35, 39)), ((4, 36, 4), (11, 39, 45)), ((0, 4, 4), (3, 35, 11))],
                             [((12, 14, 16), (67, 65, 71)), ((10, 14, 16), (11, 17, 19)),
                              ((12, 66, 20), (19, 71, 71))]]),
}


@pytest.fixture(scope="module")
def ctx():
    with lbx.Context(0) as c:
        yield c


@pytest.mark.parametrize("mask", ["reference", "fine"])
@pytest.mark.parametrize("name", CASES)
def test_fine_step_equals_oracle(ctx, name, mask):
    dims, refined = CASES[name]
    levels = [workloads.chop(dims, 32)] + refined
    masks = masks_for(mask, levels)
    rho, u = workloads.random_state(dims, 11, 1e-2, 0.02)
    ref = run_oracle(dims, levels, masks, 0.8, rho, u, 2)
    sim = make_gpu(ctx, dims, levels, masks, 0.8, rho, u)
    sim.iterate(2)
    out = gpu_levels(sim, len(levels))
    sim.close()
    for l, (a, b) in enumerate(zip(ref, out)):
        assert_bitwise(a, b, f"level {l}")
    if mask == "reference":  # doubles the density where the fine level adds to a collided cell
        return
    sim = make_gpu(ctx, dims, levels, masks, 0.8, rho, u, precision=lbx.LBX_FP32_SHIFTED)
    sim.iterate(2)
    out = gpu_levels(sim, len(levels))
    sim.close()
    for a, b in zip(ref, out):
        assert np.abs(a - b).max() <= 4 * 8 * 40 * 2.0 ** -24 * np.abs(a).max()
