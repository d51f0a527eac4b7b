"""Density-gradient tags on domains a few cells wide in x or y: the tiled kernel
leaves most of its lanes idle there, so they take a lane per cell.  The same
cells with the thin axis along z keep the tiles' lanes busy: a domain thin in x
may take twice as long as that one at most (4 and 1 cells wide with the tiles: 3.1
and 3.3 times; a lane per cell: 1.4 and 1.2)."""
import time

import numpy as np
import pytest

from lambrex_amd import lbx, workloads
from test_gpu_regrid import criterion_numpy

pytestmark = pytest.mark.gpu


def fastest(sim, ctx):
    best = 1e30
    for _ in range(8):
        ctx.sync()
        t = time.perf_counter()
        sim.tag_cells(lbx.LBX_TAG_DENSITY_GRADIENT, 1e-3)
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("thin,wide", [((3, 850, 850), (850, 850, 3)), ((1, 1500, 1500), (1500, 1500, 1))])
def test_thin_domains_take_no_tiles(ctx, thin, wide):
    times = []
    for dims in (thin, wide):
        sim = lbx.Sim(ctx, dims)
        sim.define_level(0, [((0, 0, 0), tuple(d - 1 for d in dims))])
        sim.set_tau(0, 0.7)
        sim.init_from_fields(*workloads.plane_pulse(dims, 1e-2, axis=int(np.argmax(dims))))
        sim.iterate(3)
        times.append(fastest(sim, ctx))
        sim.close()
    assert times[0] <= 2 * times[1], times


@pytest.mark.parametrize("precision", [lbx.LBX_FP64, lbx.LBX_FP32_SHIFTED])
@pytest.mark.parametrize("dims", [(12, 130, 67), (14, 130, 67), (130, 6, 110), (130, 8, 110)])
def test_tags_on_both_sides_of_the_rule(ctx, dims, precision):
    rho, u = workloads.random_state(dims, seed=17, rho_sigma=1e-2, u_amp=0.02)
    sim = lbx.Sim(ctx, dims, precision=precision)
    sim.define_level(0, workloads.chop(dims, 64))
    sim.set_tau(0, 0.7)
    sim.init_from_fields(rho, u)
    sim.iterate(2)
    s = criterion_numpy(*sim.get_hydro(0), lbx.LBX_TAG_DENSITY_GRADIENT)
    threshold = float(np.sqrt(np.median(s)))
    tags = sim.tag_cells(lbx.LBX_TAG_DENSITY_GRADIENT, threshold)
    sim.close()
    assert np.array_equal(tags, (s > threshold * threshold).astype(np.uint8))
