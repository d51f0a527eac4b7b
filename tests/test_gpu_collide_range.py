"""The FP64 collision over the exponents of its operands, against the CPU
oracle, bitwise: the divisions share a reciprocal while the density lies within
2^-100 .. 2^100 and are the compiler's own outside it.  States of every scale
around those bounds and far from them, of either sign, with a density that
nearly cancels, at rest, empty, and with a momentum close to the smallest
number."""
import numpy as np
import pytest

from lambrex_amd import lbx, workloads
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

EXPONENTS = (-1040, -1000, -500, -102, -101, -100, -99, -3, 0, 98, 99, 100, 101, 500, 900)


def states(shape):
    rng = np.random.default_rng(41)
    n = int(np.prod(shape))
    f = np.zeros((15, n))
    for c in range(n):
        kind, e = c % 6, EXPONENTS[(c // 6) % len(EXPONENTS)]
        if kind == 0:
            v = rng.random(15) + 0.1
        elif kind == 1:
            v = rng.standard_normal(15)
        elif kind == 2:
            v = rng.random(15)
            v[0] = 2.0 ** -40 - v[1:].sum()
        elif kind == 3:
            v = np.ones(15)
        elif kind == 4:
            v = np.zeros(15)
        else:
            v = np.zeros(15)
            v[0], v[1] = 1.0, 2.0 ** -1000
        f[:, c] = np.ldexp(v, e)
    return f.reshape((15,) + shape)


@pytest.mark.parametrize("tau_b", [0.8, 0.6])
def test_collision_bitwise_over_exponents(tau_b):
    dims = (16, 9, 10)
    boxes = workloads.chop(dims, 32)
    f = states(dims[::-1])
    o = orc.Sim(*dims, 0.8, tau_b, boxes=[(list(a), list(b)) for a, b in boxes])
    o.set_f(f)
    o.iterate(1)
    ref = o.get_f()
    o.close()
    number = ~np.isnan(ref)  # an empty cell's velocity is 0 / 0, and a NaN's bits are not defined
    assert number.mean() > 0.5
    with lbx.Context(0) as ctx:
        sim = lbx.Sim(ctx, dims)
        sim.define_level(0, boxes)
        sim.set_tau(0, 0.8, tau_b)
        sim.set_f(f)
        sim.iterate(1)
        out = sim.get_f()
        sim.close()
    assert np.array_equal(~np.isnan(out), number)
    assert np.array_equal(out[number].view(np.uint64), ref[number].view(np.uint64))
