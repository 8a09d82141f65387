"""The direct kernels where their blocks end: channel counts that fill no block, tap rows taken in
one, several or single pieces, every block size, sums cut into chunks that run across samples.

Bounds: float32 sums of at most some 10^5 products with relative error 2^-24 each, whose errors add
like a random walk (10^2.5 * 6e-8 = 2e-5) on results of the size of the largest terms; bfloat16
storage of the intermediate tensor alone gives 2^-9, about 8 of them in a chain 2e-2."""

import pytest
import torch

from deconver_amd import _lib, ops
from oracle import ndc_oracle as O
from tests.helpers import hostcheck_library, make_case

# (C, groups, sc, kernel, spatial, batch)
SMALL = [
    (5, 1, 7, (3, 3, 3), (4, 5, 6), 2),      # 8-blocks with rows of padding, three loops of taps
    (9, 3, 5, (3, 3), (7, 9), 3),
    (3, 1, 3, (9,), (41,), 2),               # a row of 9 taps in three pieces
    (2, 1, 5, (7,), (50,), 2),               # ... of 7 in single taps
    (4, 2, 3, (5, 3, 5), (5, 4, 7), 2),
    # (one tap needs two sources: with one, s cancels out of s n / d, and the bound above is on sums
    # next to which the true gradient of z, zero, has no size)
    (3, 3, 3, (1, 1, 1), (3, 4, 5), 2),
    (4, 2, 4, (3, 3, 1), (3, 5, 1), 2),
    (2, 1, 2, (3, 3, 3), (1, 1, 1), 1),      # every tap but one outside
    (4, 2, 2, (3, 3, 3), (14, 15, 16), 3),   # several chunks, their runs crossing samples
]
# wide enough for the largest blocks of output channels
LARGE = [
    (8, 1, 8, (3, 3, 3), (40, 60, 60), 1),
    (5, 1, 8, (5, 5), (370, 371), 1),
    (2, 1, 12, (3, 3, 3), (30, 40, 61), 2),
]
TOL = {torch.float32: 2e-5, torch.bfloat16: 2e-2}


def _compare(lib, geom, dtype, device):
    C, G, sc, ks, sp, B = geom
    m = C // G
    x, z, h, bias, gout = make_case(C, G, sc, ks, sp, B=B, dtype=dtype, bias_shift=0.3, device=device)
    kw = dict(groups=G, m=m, sc=sc, eps=1e-16, relu_input=True, path=_lib.PATH_DIRECT)
    out, t1 = ops.update_forward(lib, x, z, h, bias, **kw)
    grads = ops.update_backward(lib, x, z, t1, h, bias, gout, **kw)
    d = [t.detach().cpu().double() for t in (x, z, h, bias, gout)]
    ro, rt1 = O.update_grouped(d[0], d[1], d[2], d[3], G, m, sc, 1e-16, True)
    ref = (ro, rt1, *O.update_backward(*d, G, m, sc, 1e-16, True))
    errs = [O.rel_err(a.detach().cpu(), b) for a, b in zip((out, t1, *grads), ref)]
    assert all(e < TOL[dtype] for e in errs), (geom, dtype, errs)


@pytest.mark.parametrize("geom", SMALL)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_blocks_on_the_host_build(geom, dtype):
    _compare(hostcheck_library(), geom, dtype, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("geom", SMALL + LARGE)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_blocks_on_the_gpu(geom, dtype):
    print("case", geom, dtype, flush=True)
    _compare(_lib.get_library(), geom, dtype, "cuda")
