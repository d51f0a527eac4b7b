"""Every kernel of the two-step pass (tests/pair_paths.py) against single passes,
and the 256^3 lattice between walls that the benchmark steps: same bits."""
import numpy as np
import pytest

from lambrex_amd import lbx, workloads
from pair_paths import CASES
from test_gpu_pair import start

pytestmark = pytest.mark.gpu


def fields(sim):
    return np.concatenate([a.reshape(-1) for part in sim.hydro_level(0) for a in part])


@pytest.mark.parametrize("dims,periodic,precision", [c[:3] for c in CASES] + [((256, 256, 256), (1, 1, 0), lbx.LBX_FP64)])
def test_two_step_kernels_equal_single_passes(ctx, dims, periodic, precision):
    rho, u = workloads.random_state(dims, 5, 1e-2, 0.03)
    out = []
    for chunks in ((6,), (1,) * 6):
        sim = start(ctx, dims, periodic, precision, rho, u)
        ctx.profile_enable()
        for n in chunks:
            sim.iterate(n)
        launches = ctx.profile_read()[1]
        ctx.profile_enable(False)
        assert launches == (3 if len(chunks) == 1 else 5)  # two pairs and a single pass after the collide-only one
        out.append(sim.get_f() if dims[0] < 256 else fields(sim))
        sim.close()
    assert np.array_equal(out[0].view(np.uint64), out[1].view(np.uint64))
