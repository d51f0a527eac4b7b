"""The measured per-step traffic that bench.py reports beside its two- and
three-level lines: on file, and counted for the same workloads."""
import json
import sys
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))

import bench  # noqa: E402


def cells(boxes):
    return sum(int(np.prod([hi[d] - lo[d] + 1 for d in range(3)])) for lo, hi in boxes)


def state_cells_per_step(levels):
    """Cells of the populations that a level-0 step reads and writes, once per
    pass: level 0 by one pass, a level with a child by one for each of its 2^l
    steps, the finest by one for each two of them."""
    last = len(levels) - 1
    return sum((2 ** (last - 1) if l == last else 2 ** l) * cells(b) for l, b in enumerate(levels))


def test_fused_step_traffic_entries_match_the_workloads():
    dims2, cboxes, fboxes, *_ = bench.two_level_geometry()
    dims3, levels3, *_ = bench.three_level_geometry()
    for key, dims, levels in (("two_level_fused_step", dims2, [cboxes, fboxes]),
                              ("three_level_fused_step", dims3, levels3)):
        names = ["128^3"]
        for l, boxes in enumerate(levels[1:], 1):
            lo = [min(b[0][d] for b in boxes) for d in range(3)]
            hi = [max(b[1][d] for b in boxes) for d in range(3)]
            names.append("x".join(str(h - a + 1) for a, h in zip(lo, hi)))
        assert tuple(dims) == (128, 128, 128)
        t = bench.step_traffic(key, " + ".join(names))
        assert t is not None, (key, names)
        assert t["algorithmic_bytes_per_step"] == 240 * state_cells_per_step(levels)
        # a pass reads its level's state and writes it, so no fewer bytes
        assert t["over_algorithmic"] > 1.0
        assert abs(t["bytes_per_step"] / t["algorithmic_bytes_per_step"] - t["over_algorithmic"]) < 1e-3
        assert (ROOT / t["source"]).is_file()
        assert f"**{t['bytes_per_step'] / 1e6:,.0f} MB moved" in (ROOT / t["source"]).read_text(), key


def test_bench_reads_the_fused_entries():
    """The keys and workloads guarded above are the ones the lines read."""
    text = (ROOT / "bench.py").read_text()
    for key in ("two_level_fused_step", "three_level_fused_step"):
        (workload,) = json.loads(bench.TRAFFIC_FILE.read_text())[key]
        assert f'step_traffic("{key}", "{workload}")' in text
