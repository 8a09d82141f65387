"""The direct kernels' convolutions from boxes in LDS: boxes that end outside the volume, one and two rows a thread,
channels staged in several groups, blocks of output channels with padding, taps by fives, filters deep in the first axis,
planes; and a filter without boxes that takes its weights from LDS.  Oracle and bounds as in the tests of the blocks."""

import pytest
import torch

from deconver_amd import _lib
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
