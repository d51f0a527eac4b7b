"""The library's host code on failing allocations and in its copies, on a stand-in
HIP runtime (tests/cpp/fake_hip.cpp) in a process of its own: no GPU."""
import subprocess
import sys
import textwrap
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
FAKE = ROOT / "tests" / "cpp" / "_bin" / "libfake_hip.so"

PRELUDE = f"""
import ctypes, sys
sys.path.insert(0, {str(ROOT)!r})
fake = ctypes.CDLL({str(FAKE)!r}, mode=ctypes.RTLD_GLOBAL)
import numpy as np
from lambrex_amd import lbx
ctx = lbx.Context(0)
"""


def run(code):
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code)], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_a_level_whose_allocation_fails_is_not_defined():
    """Every allocation of a level's definition fails once.  The call reports
    it, and the levels that were there step on as before: a level that a failed
    call left behind would be stepped without its parent's mask."""
    run("""
    for old in (False, True):  # with and without a level to replace
        failures = 0
        while True:
            sim = lbx.Sim(ctx, (16, 16, 16))
            sim.define_level(0, [((0, 0, 0), (15, 15, 15))])
            sim.define_level(1, [((8, 8, 8), (23, 23, 23))])
            if old:
                sim.define_level(2, [((24, 24, 24), (31, 31, 31))])
            for l in range(3 if old else 2):
                sim.set_tau(l, 0.8)
            fake.fake_fail_malloc(failures + 1)
            try:
                sim.define_level(2, [((20, 20, 20), (43, 43, 43))])
                break
            except lbx.LbxError:
                failures += 1
            finally:
                fake.fake_fail_malloc(0)
            fake.fake_reset()
            sim.iterate(1)  # level 1 once as the finest level, or twice and level 2 twice
            assert fake.fake_launches(b"k_fine_step") == (4 if old else 1), failures
            sim.close()
        assert failures >= 8, failures
    """)


def test_small_read_backs_are_direct():
    """A level's fields of 2.2 and 3.5 MB (41^3, 48^3) come in two copies, those of
    4 MB and more in chunks of 1 MB: below, the threads that empty the chunks
    cost what they bring."""
    run("""
    for dims, chunks in (((41, 41, 41), 2), ((48, 48, 48), 2), ((50, 50, 50), 4), ((60, 60, 60), 7), ((64, 64, 64), 4)):
        sim = lbx.Sim(ctx, dims)
        sim.define_level(0, [((0, 0, 0), tuple(d - 1 for d in dims))])
        fake.fake_reset()
        sim.hydro_level(0)
        n = fake.fake_copies_to_host()
        assert n == chunks, (dims, n)
        sim.close()
    """)
