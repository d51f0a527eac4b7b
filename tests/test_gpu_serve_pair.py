"""Served runs advanced two steps at a time (the batch holds enough cells for
it): each run's populations equal the run alone, bit for bit.  Shapes at the
edges of a work item's column (rows of one and of several, remainders in x and
y, one plane, z-chunks with a remainder), odd and even step counts, one step,
in one drain and in odd progress calls that mix launches of one and two."""
import numpy as np
import pytest

from lambrex_amd import lbx
from test_gpu_serving import alone_plain, bitwise_equal

pytestmark = pytest.mark.gpu

MIX = [  # dims, steps, tau, amplitude
    ((96, 96, 96), 6, 0.6, 1e-2),  # with the others more cells than a launch of two steps asks for
    ((32, 33, 9), 5, 0.55, 1e-2),
    ((48, 47, 17), 4, 1.2, 3e-3),
    ((17, 24, 1), 7, 0.8, 1e-4),
    ((250, 6, 34), 3, 0.9, 5e-3),
    ((1, 65, 40), 2, 0.9, 5e-3),
    ((20, 16, 12), 1, 1.5, 2e-3),
    ((97, 34, 33), 8, 0.7, 1e-3),
]


@pytest.mark.parametrize("chunk", [0, 3])
@pytest.mark.parametrize("precision", [lbx.LBX_FP32_SHIFTED, lbx.LBX_FP64])
def test_paired_steps_equal_each_run_alone(precision, chunk):
    assert sum(int(np.prod(m[0])) for m in MIX[:1]) >= 640 << 10
    with lbx.Context(0) as ctx:
        srv = lbx.Server(ctx, precision=precision, arena_bytes=2 << 30)
        outs = []
        for dims, steps, tau, amp in MIX:
            outs.append(srv.submit(dims, steps, tau, amplitude=amp, axis=0, want_f=True)[1])
        if chunk:
            for _ in range(8):
                srv.progress(chunk)
        srv.drain()
        assert len(srv.poll()) == len(MIX)
        srv.close()
        for (dims, steps, tau, amp), o in zip(MIX, outs):
            assert bitwise_equal(o["f"], alone_plain(ctx, dims, steps, tau, amp, precision)), (dims, steps)
