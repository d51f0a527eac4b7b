"""Large read-backs (through pinned chunks and several threads) against small
ones (direct copies): a level's fields in one call equal those of its boxes,
and a whole-domain box's populations equal the same cells read in boxes.
Totals just below and at each chunk size's start, and with remainders."""
import numpy as np
import pytest

from lambrex_amd import lbx, workloads

pytestmark = pytest.mark.gpu


def make(ctx, dims, boxes, rho, u):
    sim = lbx.Sim(ctx, dims)
    sim.define_level(0, boxes)
    sim.set_tau(0, 0.8)
    sim.init_from_fields(rho, u)
    sim.iterate(3)
    return sim


@pytest.mark.parametrize("dims", [(64, 32, 31), (64, 32, 32), (37, 41, 53), (64, 64, 63), (64, 64, 64), (61, 97, 83),
                                  (128, 128, 127), (128, 128, 128), (130, 131, 149)])
def test_level_fields_equal_box_fields(dims):
    rho, u = workloads.random_state(dims, 3, 1e-2, 0.03)
    with lbx.Context(0) as ctx:
        sim = make(ctx, dims, workloads.chop(dims, 16), rho, u)
        bulk = sim.hydro_level(0)
        for b, (r, v) in enumerate(bulk):
            r1, v1 = sim.hydro(0, b)
            assert np.array_equal(r, r1) and np.array_equal(v, v1)
        sim.close()


@pytest.mark.parametrize("dims", [(20, 21, 22), (44, 40, 40), (80, 85, 90)])
def test_populations_equal_box_populations(dims):
    rho, u = workloads.random_state(dims, 4, 1e-2, 0.03)
    with lbx.Context(0) as ctx:
        out = []
        for cut in (128, 16):
            sim = make(ctx, dims, workloads.chop(dims, cut), rho, u)
            out.append(sim.get_f())
            sim.close()
    assert np.array_equal(out[0], out[1])
