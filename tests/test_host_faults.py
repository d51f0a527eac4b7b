"""The library's host code on failing allocations, its copies and launches, on a stand-in
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


def test_read_backs_come_in_few_chunks():
    """A level's fields below 2 MB (40^3) come in two copies, above in chunks of 1
    MB and from 8 MB on (64^3) of 2 MB: smaller ones leave the threads that empty
    them waiting for the next."""
    run("""
    for dims, chunks in (((40, 40, 40), 2), ((41, 41, 41), 3), ((48, 48, 48), 4), ((60, 60, 60), 7), ((64, 64, 64), 4)):
        sim = lbx.Sim(ctx, dims)
        sim.define_level(0, [((0, 0, 0), tuple(d - 1 for d in dims))])
        fake.fake_reset()
        sim.hydro_level(0)
        n = fake.fake_copies_to_host()
        assert n == chunks, (dims, n)
        sim.close()
    """)


def test_served_batches_take_the_faster_launch():
    """Batches of served runs for which two launches of one step are the faster
    take no launch of two, and the other way round."""
    run("""
    cases = [(lbx.LBX_FP32_SHIFTED, (80, 80, 80), 2, False), (lbx.LBX_FP32_SHIFTED, (200, 200, 8), 3, False),
             (lbx.LBX_FP32_SHIFTED, (300, 300, 4), 23, False), (lbx.LBX_FP64, (200, 200, 8), 3, False),
             (lbx.LBX_FP64, (8, 8, 3000), 14, False), (lbx.LBX_FP32_SHIFTED, (97, 97, 97), 1, True),
             (lbx.LBX_FP32_SHIFTED, (130, 130, 30), 5, True), (lbx.LBX_FP64, (200, 200, 8), 25, True),
             (lbx.LBX_FP64, (161, 33, 47), 11, True), (lbx.LBX_FP32_SHIFTED, (32, 32, 32), 30, True)]
    for precision, dims, runs, pairs in cases:
        srv = lbx.Server(ctx, precision=precision, arena_bytes=3 << 30)
        for _ in range(runs):
            srv.submit(dims, 5, 0.7)
        fake.fake_reset()
        srv.drain()
        assert len(srv.poll()) == runs
        srv.close()
        assert (fake.fake_launches(b"k_serve_pair") > 0) == pairs, (precision, dims, runs)
        assert fake.fake_launches(b"k_serve_step") == (0 if pairs else 6), (precision, dims, runs)
    """)


def test_refined_levels_take_the_kernel_for_their_boxes():
    """Small boxes run workgroups of 256 lanes, several to a CU, where the large
    kernels would leave most of their lanes idle."""
    run(f"""
    sys.path.insert(0, {str(ROOT / 'tests')!r})
    from fine_kernels import CASES
    from lambrex_amd import workloads
    for name, (dims, refined, lanes) in CASES.items():
        for precision, letter in ((lbx.LBX_FP64, "d"), (lbx.LBX_FP32_SHIFTED, "f")):
            sim = lbx.Sim(ctx, dims, precision=precision)
            sim.define_level(0, workloads.chop(dims, 32))
            for l, boxes in enumerate(refined):
                sim.define_level(l + 1, boxes)
            for l in range(len(refined) + 1):
                sim.set_tau(l, 0.8)
            fake.fake_reset()
            sim.iterate(1)
            for role, flag in (("finest", 1), ("middle", 0)):
                for n in (256, 512, 768):
                    ran = sum(fake.fake_launches(f"k_fine_stepI{{letter}}Lb{{flag}}{{m}}Lb{{avg}}ELi{{n}}E".encode())
                              for m in ("ELb0ELb0E", "ELb1ELb1E") for avg in (0, 1))
                    want = role in lanes and lanes[role][precision] == n
                    assert (ran > 0) == want, (name, letter, role, n, ran)
            sim.close()
    """)


def test_small_fp32_lattices_take_the_faster_pass():
    """Blocks of 6x6x6 cells, two to a CU, only where single passes take longer."""
    run("""
    cases = [((90, 15, 63), (1, 1, 0), False), ((494, 25, 5), (0, 1, 1), False), ((199, 15, 30), (1, 1, 1), False),
             ((64, 36, 36), (1, 1, 1), False), ((48, 48, 48), (0, 0, 0), True), ((48, 48, 48), (1, 1, 1), True),
             ((36, 36, 72), (1, 1, 1), True), ((11, 369, 11), (1, 1, 1), True), ((257, 28, 5), (0, 0, 0), True)]
    for dims, periodic, blocks in cases:
        sim = lbx.Sim(ctx, dims, precision=lbx.LBX_FP32_SHIFTED, periodic=periodic)
        sim.define_level(0, [((0, 0, 0), tuple(d - 1 for d in dims))])
        sim.set_tau(0, 0.8)
        sim.iterate(1)
        fake.fake_reset()
        sim.iterate(6)
        assert fake.fake_launches(b"k_step_block") == (3 if blocks else 0), (dims, periodic)
        sim.close()
    """)


def test_lattices_run_each_two_step_kernel():
    """The lattices of tests/pair_paths.py take the kernels they are listed for."""
    run(f"""
    sys.path.insert(0, {str(ROOT / 'tests')!r})
    from pair_paths import CASES
    for dims, periodic, precision, column in CASES:
        sim = lbx.Sim(ctx, dims, precision=precision, periodic=periodic)
        sim.define_level(0, [((0, 0, 0), tuple(d - 1 for d in dims))])
        sim.set_tau(0, 0.8)
        sim.iterate(1)
        fake.fake_reset()
        sim.iterate(4)
        walls = 0 if all(periodic) else 1
        for b in (0, 32, 64):
            part = f"k_step_pairI{{'df'[precision]}}Li{{b}}ELi{{(0, 16, 8)[(0, 32, 64).index(b)]}}ELb{{walls}}E"
            assert fake.fake_launches(part.encode()) == (2 if b == column else 0), (dims, precision, b)
        sim.close()
    """)
