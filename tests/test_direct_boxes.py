"""The direct kernels' convolutions from boxes in LDS: boxes that end outside the volume, one and two rows a thread,
channels staged in several groups, blocks of output channels with padding, taps by fives, filters deep in the first axis,
planes; and a filter without boxes that takes its weights from LDS.  Oracle and bounds as in the tests of the blocks."""

import pytest
import torch

from deconver_amd import _lib, ops
from tests.helpers import host_faults, hostcheck_library
from tests.test_direct_blocks import _compare

# (C, groups, sc, kernel, spatial, batch)
GEOMS = [
    (4, 2, 8, (3, 3, 3), (5, 7, 9), 1),       # one row a thread
    (6, 2, 5, (3, 3, 3), (11, 13, 19), 2),    # ragged in every direction, blocks with padding
    (2, 2, 1, (3, 3, 3), (24, 17, 33), 2),    # two rows a thread, a last row of one
    (24, 2, 20, (3, 3, 3), (6, 7, 8), 1),     # several groups of channels
    (8, 4, 4, (5, 5, 5), (7, 6, 11), 1),      # rows of 20 weights; groups of channels
    (3, 3, 3, (5, 5, 5), (4, 3, 2), 2),       # a volume smaller than the filter
    (4, 2, 3, (7, 3, 3), (9, 5, 6), 1),       # more taps in the first axis
    (4, 2, 6, (1, 5, 5), (3, 9, 10), 1),      # none there
    (6, 3, 4, (3, 3), (19, 70), 2),           # a plane; rows of more than a wavefront
    (2, 1, 2, (5, 5), (1, 300), 1),           # a single row
]
LARGE = [(32, 8, 8, (3, 3, 3), (40, 41, 43), 1), (16, 16, 2, (3, 3), (131, 517), 4)]
STAGED = [(16, 16, 4, (7, 7), (64, 64), 8)]


@pytest.mark.parametrize("geom", GEOMS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_boxes_on_the_host_build(geom, dtype):
    lib = hostcheck_library()
    _compare(lib, geom, dtype, "cpu")
    assert host_faults(lib)[0] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("geom", GEOMS + LARGE + STAGED)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_boxes_on_the_gpu(geom, dtype):
    print("case", geom, dtype, flush=True)
    _compare(_lib.get_library(), geom, dtype, "cuda")


# filters of unequal extents and images beyond the boxes: one position at a time, three and five taps, the weights from the
# scalar unit and from LDS
UNEQUAL = [(4, 2, 6, (5, 3), (9, 11), 1), (6, 3, 4, (3, 5, 3), (5, 6, 7), 2), (4, 2, 3, (3, 5), (8, 12), 1)]
WITHOUT = [(4, 2, 6, (3, 3), (384, 256), 1), (16, 16, 4, (3, 3), (384, 256), 2), (16, 16, 4, (5, 3), (64, 64), 8)]


@pytest.mark.parametrize("geom", UNEQUAL)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_one_position_at_a_time_on_the_host_build(geom, dtype):
    lib = hostcheck_library()
    _compare(lib, geom, dtype, "cpu")
    assert host_faults(lib)[0] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("geom", UNEQUAL + WITHOUT)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_one_position_at_a_time_on_the_gpu(geom, dtype):
    print("case", geom, dtype, flush=True)
    _compare(_lib.get_library(), geom, dtype, "cuda")


def _box(sp, ks=(3, 3, 3), nin=1, nb=4, cin=4, units=16):
    """(boxes looked at, workgroups, threads, rows a thread) of a launch; no workgroups: no box."""
    import ctypes

    lib = hostcheck_library()
    like = torch.empty(1, 8, *sp, device="meta")
    g = ops.make_geom_for(like, torch.empty(8, 8, *ks, device="meta"), 2, 4, 8, 1e-16, True)
    launch = (ctypes.c_longlong * 3)()
    lib._dll.ndc_host_box.restype = ctypes.c_longlong
    looked = lib._dll.ndc_host_box(ctypes.byref(g), nin, nb, cin, ctypes.c_longlong(units), launch)
    return looked, *launch


def test_a_size_is_searched_once():
    """What the host does for a launch: few boxes looked at, none where none can be, and none for a size it has seen."""
    sizes = [(20 + k, 24 + k, 22 + 2 * k) for k in range(24)]
    first = [_box(sp, nin=nin)[0] for sp in sizes for nin in (1, 2, 3)]
    assert all(0 < n <= 800 for n in first)
    assert not any(_box(sp, nin=nin)[0] for sp in sizes for nin in (1, 2, 3))
    for sp, ks in (((160, 160, 160), (3, 3, 3)), ((192, 192, 192), (3, 3, 3)), ((320, 320), (3, 3))):
        assert _box(sp, ks)[:2] == (0, 0)


def test_boxes_of_fewer_threads_than_a_launch_takes():
    """46 x 1 x 60 positions a unit are 2816 threads one at a time and more in boxes: those reach 2^32 at fewer units."""
    sp, ks, most = (46, 1, 60), (7, 3, 3), (2 ** 32 - 1) // 2816
    for units in (1000, most // 2, most * 9 // 10, most):
        _, groups, threads, _ = _box(sp, ks, 1, 1, 1, units)
        assert groups * threads < 2 ** 32 and (groups > 0) == (units < most)
