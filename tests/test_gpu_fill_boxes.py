"""A new level's cells are looked up among the boxes that meet its own: with
few of them, and with more than a workgroup lists, as old boxes of a remake
and as the parent's boxes of a fill, against the piecewise-constant rule."""
import numpy as np
import pytest

from lambrex_amd import lbx, workloads
from test_gpu_twolevel import fine_boxes_in

pytestmark = pytest.mark.gpu


def up(a):
    for axis in (1, 2, 3):
        a = np.repeat(a, 2, axis=axis)
    return a


@pytest.mark.parametrize("precision", [lbx.LBX_FP64, lbx.LBX_FP32_SHIFTED])
@pytest.mark.parametrize("cut", [2, 6, 18])
def test_remake_and_fill_take_the_box_that_holds_the_cell(precision, cut):
    dims = (16, 16, 16)
    rho, u = workloads.random_state(dims, 3, 1e-2, 0.03)
    many = fine_boxes_in((6, 6, 6), (23, 23, 23), cut)  # 729, 27 or 1
    with lbx.Context(0) as ctx:
        sim = lbx.Sim(ctx, dims, precision=precision)
        sim.define_level(0, workloads.chop(dims, 8))
        sim.set_tau(0, 0.8)
        sim.init_from_fields(rho, u)
        sim.define_level(1, many)
        sim.set_tau(1, 1.1)
        sim.fill_from_coarse(1)
        sim.set_fine_mask(many)
        sim.iterate(2)
        coarse, old = sim.get_f(0), sim.get_f_bbox(1)[0]
        sim.define_level(2, fine_boxes_in((14, 14, 14), (45, 45, 45), 16))
        sim.fill_from_coarse(2)
        assert np.array_equal(sim.get_f_bbox(2)[0], up(old)[:, 2:34, 2:34, 2:34])
        sim.clear_level(2)
        sim.remake_level(1, [((4, 4, 4), (25, 15, 25)), ((4, 16, 4), (25, 25, 25))])
        new = sim.get_f_bbox(1)[0]
        sim.close()
    want = up(coarse[:, 2:13, 2:13, 2:13])
    want[:, 2:20, 2:20, 2:20] = old
    assert np.array_equal(new, want)
