"""The direct kernels with a unit's weights in LDS: wavefronts just short of and at the rule's limits (both
convolutions on either side, and one on each), padded channel blocks, taps by fives, and filters too large for
it.  Oracle and bounds as in the tests of their blocks."""

import pytest
import torch

from deconver_amd import _lib
from tests.helpers import hostcheck_library
from tests.test_direct_blocks import _compare

GEOMS = [
    (767, 767, 8, (3, 3, 3), (5, 5, 6), 1),      # K 3068 wavefronts, A 3068 of 8 outputs: the scalar unit
    (768, 768, 8, (3, 3, 3), (5, 5, 6), 1),      # one group more: LDS
    (512, 128, 3, (5, 5), (12, 13), 6),          # K in LDS, A (12 288) not; a channel of padding
    (128, 64, 5, (3, 3), (13, 15), 24),          # eights with three of padding
]
# 19 and 8 channels with 8 outputs at a time: 8 x 19 x 27 = 4104 weights are more than LDS is given, 8 x 8 x 27 fit
LARGE = [(8, 1, 19, (3, 3, 3), (48, 48, 48), 1), (19, 1, 8, (3, 3, 3), (48, 48, 48), 1), (8, 2, 8, (3, 3, 3), (47, 50, 49), 1)]


@pytest.mark.parametrize("geom", GEOMS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_staged_on_the_host_build(geom, dtype):
    _compare(hostcheck_library(), geom, dtype, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("geom", GEOMS + LARGE)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_staged_on_the_gpu(geom, dtype):
    print("case", geom, dtype, flush=True)
    _compare(_lib.get_library(), geom, dtype, "cuda")
