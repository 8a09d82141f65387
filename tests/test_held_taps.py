"""2-D forwards of small launches: widths that fill no wavefront, images of few rows, several tiles a row,
and one of many images, against the oracle in float64.  Bounds as in the other parity tests."""

import pytest
import torch

from deconver_amd import _lib, ops
from oracle import ndc_oracle as O
from tests.helpers import hostcheck_library, make_case

# (C, kernel, spatial, batch)
GEOMS = [(3, (5, 5), (1, 7), 2), (2, (5, 5), (2, 1), 1), (4, (5, 5), (33, 127), 1), (2, (3, 3), (50, 64), 1),
         (5, (3, 3), (19, 65), 2), (2, (5, 5), (37, 200), 1), (3, (5, 5), (20, 301), 1)]
PAST = [(520, (5, 5), (64, 30), 1)]          # more workgroups than the chip holds at once
TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2}


def _compare(lib, geom, dtype, device):
    C, ks, sp, B = geom
    x, z, h, bias, _ = make_case(C, C, 4, ks, sp, B=B, dtype=dtype, bias_shift=0.3, device=device)
    kw = dict(groups=C, m=1, sc=4, eps=1e-16, relu_input=True, path=_lib.PATH_FUSED)
    out, t1, (sd, nd) = ops.update_forward(lib, x, z, h, bias, save_ratio=True, **kw)
    d = [t.detach().cpu().double() for t in (x, z, h, bias)]
    ro, rt1 = O.update_grouped(d[0], d[1], d[2], d[3], C, 1, 4, 1e-16, True)
    den = O.op_A(rt1, d[2], C, 1, 4) + 1e-16
    ref = (ro, rt1, O.rectified_source(d[1], d[3], True) / den, (O.op_A(d[0], d[2], C, 1, 4) + 1e-16) / den)
    errs = [O.rel_err(a.detach().cpu(), b) for a, b in zip((out, t1, sd, nd), ref)]
    assert all(e < TOL[dtype] for e in errs), (geom, dtype, errs)


@pytest.mark.parametrize("geom", GEOMS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_forward_on_the_host_build(geom, dtype):
    lib = hostcheck_library()
    _compare(lib, geom, dtype, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("geom", GEOMS + PAST)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_forward_on_the_gpu(geom, dtype):
    print("case", geom, dtype, flush=True)
    _compare(_lib.get_library(), geom, dtype, "cuda")
