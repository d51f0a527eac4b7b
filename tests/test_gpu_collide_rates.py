"""The FP64 collision at relaxation rates up to the largest number, which
set_relax accepts, against the CPU oracle: a trace that relaxes to infinity makes
populations infinite or undefined exactly where the reference's arithmetic does."""
import numpy as np
import pytest

from lambrex_amd import lbx, workloads
from oracle import oracle as orc
from test_gpu_collide_range import states

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("omega_s,omega_b", [(0.8, 2.0 ** 1000), (0.8, -1.7e308), (2.0 ** 54, 0.8)])
def test_collision_over_rates(omega_s, omega_b):
    dims = (16, 9, 10)
    f = states(dims[::-1])
    cells = f.reshape(15, -1)
    after = np.stack([orc.collide_cell(cells[:, c], omega_s, omega_b) for c in range(cells.shape[1])], axis=1)
    ref = orc.stream_periodic(after.reshape(f.shape))
    number = ~np.isnan(ref)
    with lbx.Context(0) as ctx:
        sim = lbx.Sim(ctx, dims)
        sim.define_level(0, workloads.chop(dims, 32))
        sim.set_relax(0, omega_s, omega_b)
        sim.set_f(f)
        sim.iterate(1)
        out = sim.get_f()
        sim.close()
    assert np.array_equal(~np.isnan(out), number)
    assert np.array_equal(out[number].view(np.uint64), ref[number].view(np.uint64))
