"""Hierarchies whose refined levels run each of the kernels of k_fine_step: the
small one (tiles of at most 256 cells a plane) and the large ones."""
from lambrex_amd import workloads


def slab(extents, cut, lo):
    return [(tuple(a + o for a, o in zip(blo, lo)), tuple(a + o for a, o in zip(bhi, lo)))
            for blo, bhi in workloads.chop(extents, cut)]


def two(cut):
    return (72, 72, 72), [slab((64, 128, 128), cut, (40, 8, 8))]


CASES = {  # name: (coarse extents, boxes of each refined level, lanes per workgroup: FP64 and FP32, finest and middle)
    "boxes_of_8": two(8) + ({"finest": (256, 256)},),
    "boxes_of_16": two(16) + ({"finest": (512, 256)},),
    "one_box_each": ((64, 64, 64), [slab((64, 96, 96), 64, (32, 16, 16)), slab((64, 128, 128), 64, (96, 64, 64))],
                     {"finest": (512, 768), "middle": (256, 512)}),
}
