"""The marching kernels on 2-D problems, which serve images past the lines of the one-shot kernels: rows of
one, part of one and several wavefronts, single columns and column pairs (even widths from 128 on), one
to three segments of the march, ragged last ones, with and without the kept ratios, against the oracle in
float64.  On the host build small images are sent down the march, and every access of LDS is checked.  Bounds as in
the other parity tests."""

import pytest
import torch

from deconver_amd import _lib, ops
from oracle import ndc_oracle as O
from tests.helpers import host_faults, host_march, hostcheck_library, make_case

# (C, kernel, spatial, batch)
GEOMS = [(3, (5, 5), (9, 12), 2), (2, (5, 5), (3, 70), 1), (2, (3, 3), (7, 9), 2), (2, (5, 5), (70, 12), 1), (1, (5, 5), (101, 6), 2),
         (3, (5, 5), (1, 7), 2), (2, (5, 5), (2, 1), 1), (4, (5, 5), (33, 127), 1), (2, (3, 3), (50, 64), 1), (2, (3, 3), (19, 65), 2),
         (1, (5, 5), (9, 128), 2), (1, (3, 3), (40, 130), 1), (1, (5, 5), (37, 200), 1), (1, (5, 5), (20, 301), 1)]
# past the lines: the forward by pairs and by single columns, the backward by both
LARGE = [(64, (5, 5), (162, 166), 1), (64, (5, 5), (163, 163), 1), (40, (3, 3), (150, 152), 2), (60, (3, 3), (120, 127), 2)]
TOL = {torch.float32: (1e-5, 1e-4), torch.bfloat16: (2e-2, 2e-2)}


def _compare(lib, geom, dtype, saved, relu, device):
    C, ks, sp, B = geom
    x, z, h, bias, gout = make_case(C, C, 4, ks, sp, B=B, dtype=dtype, bias_shift=0.3, positive_z=not relu, device=device)
    kw = dict(groups=C, m=1, sc=4, eps=1e-6, relu_input=relu, path=_lib.PATH_FUSED)
    out, t1, *kept = ops.update_forward(lib, x, z, h, bias, save_ratio=saved, **kw)
    got = ops.update_backward(lib, x, z, t1, h, bias, gout, saved=kept[0] if saved else None, **kw)
    d = [t.detach().cpu().double() for t in (x, z, h, bias, gout)]
    ro, rt1 = O.update_grouped(*d[:4], C, 1, 4, 1e-6, relu)
    refs = [ro, rt1]
    if saved:
        den = O.op_A(rt1, d[2], C, 1, 4) + 1e-6
        refs += [O.rectified_source(d[1], d[3], relu) / den, (O.op_A(d[0], d[2], C, 1, 4) + 1e-6) / den]
    for a, r in zip((out, t1) + (tuple(kept[0]) if saved else ()), refs):
        assert O.rel_err(a.detach().cpu(), r) < TOL[dtype][0], geom
    for a, r in zip(got, O.update_backward(*d, C, 1, 4, 1e-6, relu)):
        assert O.rel_err(a.detach().cpu(), r) < TOL[dtype][1], geom


@pytest.mark.parametrize("geom", GEOMS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("saved", [False, True])
@pytest.mark.parametrize("relu", [False, True])
def test_march_on_the_host_build(geom, dtype, saved, relu):
    lib = hostcheck_library()
    host_faults(lib)
    with host_march(lib):
        _compare(lib, geom, dtype, saved, relu, "cpu")
    n, first = host_faults(lib)
    assert n == 0, f"faults: {n} ({first})"


def test_the_two_forms_differ():
    """(in the order of their sums: the switch does something, and is back in its place)"""
    lib = hostcheck_library()
    x, z, h, bias, _ = make_case(2, 2, 4, (5, 5), (20, 30), B=1, bias_shift=0.3)
    kw = dict(groups=2, m=1, sc=4, eps=1e-6, relu_input=True, path=_lib.PATH_FUSED)
    tiles = ops.update_forward(lib, x, z, h, bias, **kw)[0]
    with host_march(lib):
        march = ops.update_forward(lib, x, z, h, bias, **kw)[0]
    assert torch.equal(tiles, ops.update_forward(lib, x, z, h, bias, **kw)[0])
    assert not torch.equal(tiles, march) and O.rel_err(tiles, march.double()) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("geom", LARGE)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_march_on_the_gpu(geom, dtype):
    print("case", geom, dtype, flush=True)
    _compare(_lib.get_library(), geom, dtype, True, True, "cuda")
