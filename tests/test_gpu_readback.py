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


@pytest.mark.parametrize("steps", [0, 3])
def test_uneven_boxes_equal_box_fields(steps):
    """A level's fields in one launch, and box by box where one large box and
    many small ones would leave it mostly idle, for a level array and patches."""
    dims = (128, 64, 40)
    large = [((0, 0, 0), (127, 63, 31))]
    small = [(tuple(a + o for a, o in zip(lo, (0, 0, 32))), tuple(a + o for a, o in zip(hi, (0, 0, 32))))
             for lo, hi in workloads.chop((128, 64, 8), 8)]
    rho, u = workloads.random_state(dims, 3, 1e-2, 0.03)
    for boxes in (small[:5] + large + small[5:], workloads.chop(dims, 24)):
        for fine in ([((8, 8, 8), (11, 19, 15)), ((12, 8, 8), (39, 39, 29)), ((8, 20, 8), (11, 39, 29))], None):
            with lbx.Context(0) as ctx:
                sim = lbx.Sim(ctx, dims)
                sim.define_level(0, boxes)
                sim.set_tau(0, 0.8)
                sim.init_from_fields(rho, u)
                if fine:
                    sim.define_level(1, fine)
                    sim.set_tau(1, 1.1)
                    sim.fill_from_coarse(1)
                if steps:
                    sim.iterate(steps)
                for level in range(2 if fine else 1):
                    for b, (r, v) in enumerate(sim.hydro_level(level)):
                        r1, v1 = sim.hydro(level, b)
                        assert np.array_equal(r, r1) and np.array_equal(v, v1)
                sim.close()
