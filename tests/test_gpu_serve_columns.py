"""Served runs advanced two steps at a time in columns of rows that are no
multiple of 16 cells: whole rows, pieces of 48 and 64 cells with a remainder.
Each run's populations equal the run alone, bit for bit."""
import pytest

from lambrex_amd import lbx
from test_gpu_serving import alone_plain, bitwise_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [lbx.LBX_FP32_SHIFTED, lbx.LBX_FP64])
@pytest.mark.parametrize("dims,runs", [((97, 97, 97), 1), ((130, 130, 30), 5), ((161, 33, 47), 11), ((17, 100, 100), 15)])
def test_ragged_columns_equal_each_run_alone(dims, runs, precision):
    with lbx.Context(0) as ctx:
        srv = lbx.Server(ctx, precision=precision, arena_bytes=4 << 30)
        first = srv.submit(dims, 6, 0.7, amplitude=5e-3, axis=0, want_f=True)[1]
        for _ in range(runs - 2):
            srv.submit(dims, 5, 0.8, amplitude=1e-3)
        last = srv.submit(dims, 5, 0.6, amplitude=1e-2, axis=0, want_f=True)[1] if runs > 1 else None
        srv.drain()
        assert len(srv.poll()) == runs
        srv.close()
        assert bitwise_equal(first["f"], alone_plain(ctx, dims, 6, 0.7, 5e-3, precision))
        if last:
            assert bitwise_equal(last["f"], alone_plain(ctx, dims, 5, 0.6, 1e-2, precision))
