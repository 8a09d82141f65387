"""Weight gradients over few voxels, in one launch without splits: voxel counts around the granules and
turns of a wavefront and at the two limits of the rule, samples, tiles cut by the result, against
float64."""

import pytest
import torch

from deconver_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
# (one wavefront's first granules; an empty last turn; every wavefront once and one over; several rounds
# with a cut turn; the limits, inside and outside; samples with cut turns)
@pytest.mark.parametrize("batch,n", [(2, 1), (2, 27), (2, 64), (1, 129), (1, 256), (1, 257), (1, 511), (1, 512), (1, 513),
                                     (4, 100), (2, 511), (1, 1024), (1, 1028), (3, 341)])
# (result of one element; cut tiles of 16; the most tiles of 16; tiles of 32, cut)
@pytest.mark.parametrize("rows,cols", [(1, 1), (17, 33), (256, 256), (272, 257), (514, 130)])
def test_weight_gradient_of_few_voxels(rows, cols, batch, n, dtype):
    print(rows, cols, batch, n, dtype, flush=True)
    gen = torch.Generator().manual_seed(rows + n)
    g = torch.randn(batch, rows, n, generator=gen).to("cuda", dtype)
    x = torch.randn(batch, cols, n, generator=gen).to("cuda", dtype)
    gw, gb = ops.weight_grad(_lib.get_library(), g, x, need_bias_grad=True)
    g64, x64 = g.cpu().double(), x.cpu().double()
    want = torch.bmm(g64, x64.transpose(1, 2).contiguous()).sum(0)
    size = torch.bmm(g64.abs(), x64.abs().transpose(1, 2).contiguous()).sum(0)   # products are exact or rounded once
    bound = (batch * n + 16) * 2.0 ** -24
    assert bool(((gw.cpu().double() - want).abs() <= bound * size + 1e-30).all())
    assert bool(((gb.cpu().double() - g64.sum((0, 2))).abs() <= bound * g64.abs().sum((0, 2)) + 1e-30).all())
    again, none = ops.weight_grad(_lib.get_library(), g, x)
    assert none is None and torch.equal(again, gw)


# the most samples of the form without splits, and one more
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch,n", [(8, 64), (9, 64), (2, 27), (3, 27), (4, 27), (5, 27), (64, 16), (128, 1)])
def test_many_samples(batch, n, dtype):
    test_weight_gradient_of_few_voxels(17, 33, batch, n, dtype)
