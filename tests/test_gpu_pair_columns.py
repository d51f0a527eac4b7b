"""Two-step passes over columns of a lattice's own width against single passes,
bit for bit: whole rows, two and three parts of a row, rows with a remainder,
thin lattices, walls on every axis."""
import numpy as np
import pytest

from lambrex_amd import lbx, workloads
from test_gpu_pair import start

pytestmark = pytest.mark.gpu

CASES = [  # dims, periodic, precision
    ((72, 72, 72), (1, 1, 1), lbx.LBX_FP64),
    ((100, 100, 100), (1, 1, 1), lbx.LBX_FP64),
    ((67, 90, 81), (0, 0, 0), lbx.LBX_FP64),
    ((85, 85, 85), (0, 1, 1), lbx.LBX_FP32_SHIFTED),
    ((48, 48, 256), (1, 1, 1), lbx.LBX_FP32_SHIFTED),
    ((10, 256, 256), (1, 1, 1), lbx.LBX_FP32_SHIFTED),
    ((20, 200, 200), (1, 0, 1), lbx.LBX_FP64),
    ((99, 60, 133), (1, 0, 0), lbx.LBX_FP32_SHIFTED),
]


@pytest.fixture(scope="module")
def ctx():
    with lbx.Context(0) as c:
        yield c


@pytest.mark.parametrize("dims,periodic,precision", CASES)
def test_own_columns_equal_single_passes(ctx, dims, periodic, precision):
    rho, u = workloads.random_state(dims, 5, 1e-2, 0.03)
    a, b = (start(ctx, dims, periodic, precision, rho, u) for _ in range(2))
    a.iterate(7)
    for _ in range(7):
        b.iterate(1)
    fa, fb = a.get_f(), b.get_f()
    a.close()
    b.close()
    assert np.array_equal(fa.view(np.uint64), fb.view(np.uint64))
