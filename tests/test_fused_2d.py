"""The one-shot kernels of small images (2-D 3x3 and 5x5 updates tile by tile): images smaller than a
tile, one pixel past a tile's rows or columns, odd and single rows and columns, several tiles to a
backward workgroup, and launches on either side of the rules that choose them, against the oracle in
float64.  Bounds as in the other parity tests."""

import pytest
import torch

from deconver_amd import _lib, ops
from oracle import ndc_oracle as O
from tests.helpers import host_faults, hostcheck_library, make_case

# (C, kernel, spatial, batch)
GEOMS = [(1, (5, 5), (1, 1), 1), (2, (5, 5), (3, 2), 1), (1, (3, 3), (2, 16), 2), (2, (5, 5), (15, 17), 1), (1, (5, 5), (17, 32), 2),
         (2, (3, 3), (33, 33), 1), (1, (5, 5), (34, 48), 1), (1, (3, 3), (50, 31), 1)]
# ... past 1024 tiles a backward workgroup takes several; 0.9 M and 1.7 M pixels are the rules' lines
LARGE = [(40, (5, 5), (96, 100), 2), (24, (3, 3), (131, 67), 4), (32, (5, 5), (167, 168), 1), (32, (5, 5), (168, 168), 1),
         (64, (5, 5), (161, 165), 1), (64, (5, 5), (163, 163), 1)]
TOL = {torch.float32: (1e-5, 1e-4), torch.bfloat16: (2e-2, 2e-2)}


def _compare(lib, geom, dtype, relu, device):
    C, ks, sp, B = geom
    x, z, h, bias, gout = make_case(C, C, 4, ks, sp, B=B, dtype=dtype, bias_shift=0.3, positive_z=not relu, device=device)
    if not relu:
        bias = None
    kw = dict(groups=C, m=1, sc=4, eps=1e-6, relu_input=relu, path=_lib.PATH_FUSED)
    out, t1, kept = ops.update_forward(lib, x, z, h, bias, save_ratio=True, **kw)
    plain = ops.update_forward(lib, x, z, h, bias, need_t1=False, **kw)[0]
    assert torch.equal(out, plain)
    got = ops.update_backward(lib, x, z, t1, h, bias, gout, saved=kept, **kw)
    d = [None if t is None else t.detach().cpu().double() for t in (x, z, h, bias, gout)]
    ro, rt1 = O.update_grouped(d[0], d[1], d[2], d[3], C, 1, 4, 1e-6, relu)
    den = O.op_A(rt1, d[2], C, 1, 4) + 1e-6
    s = O.rectified_source(d[1], d[3], relu)
    refs = (ro, rt1, s / den, (O.op_A(d[0], d[2], C, 1, 4) + 1e-6) / den)
    for a, r in zip((out, t1) + tuple(kept), refs):
        assert O.rel_err(a.detach().cpu(), r) < TOL[dtype][0], geom
    for a, r in zip(got, O.update_backward(d[0], d[1], d[2], d[3], d[4], C, 1, 4, 1e-6, relu)):
        if a is not None:
            assert O.rel_err(a.detach().cpu(), r) < TOL[dtype][1], geom
    for mask in ((1, 0, 0, 0), (0, 1, 0, 1), (0, 0, 1, 0)):
        part = ops.update_backward(lib, x, z, t1, h, bias, gout, saved=kept, need_x=bool(mask[0]), need_z=bool(mask[1]),
                                   need_h=bool(mask[2]), need_b=bool(mask[3]), **kw)
        for want, a, b in zip(mask, part, got):
            assert (a is None) == (not want or b is None)
            assert a is None or torch.equal(a, b)


@pytest.mark.parametrize("geom", GEOMS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("relu", [False, True])
def test_tiles_on_the_host_build(geom, dtype, relu):
    lib = hostcheck_library()
    host_faults(lib)
    _compare(lib, geom, dtype, relu, "cpu")
    n, first = host_faults(lib)
    assert n == 0, f"faults: {n} ({first})"


@pytest.mark.gpu
@pytest.mark.parametrize("geom", GEOMS + LARGE)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_tiles_on_the_gpu(geom, dtype):
    print("case", geom, dtype, flush=True)
    _compare(_lib.get_library(), geom, dtype, True, "cuda")


# past the lines that covered pixels and lanes draw, and on this side of them: 3x3 in tiles one way, both ways and
# neither, 5x5 of many part-empty tiles; even and odd widths that march by pairs and by single columns
LINES = [(91, (3, 3), (19, 33), 8), (64, (3, 3), (33, 33), 8), (300, (3, 3), (13, 17), 8), (35, (3, 3), (58, 65), 8),
         (40, (3, 3), (60, 130), 2), (40, (3, 3), (60, 131), 2), (281, (5, 5), (33, 34), 8), (20, (5, 5), (100, 130), 4)]


@pytest.mark.gpu
@pytest.mark.parametrize("geom", LINES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_lines_on_the_gpu(geom, dtype):
    print("case", geom, dtype, flush=True)
    _compare(_lib.get_library(), geom, dtype, True, "cuda")


def test_non_finite_sources_stay_where_they_are():
    """A NaN and an infinity in z at a corner and on a tile's edge reach exactly the entries of every
    result that the oracle's arithmetic carries them to."""
    C, ks, sp = 1, (5, 5), (19, 35)
    lib = hostcheck_library()
    x, z, h, bias, gout = make_case(C, C, 4, ks, sp, B=1, bias_shift=0.3)
    z[0, 1, 0, 0], z[0, 2, 15, 31], z[0, 0, 18, 34] = float("nan"), float("inf"), float("nan")
    kw = dict(groups=C, m=1, sc=4, eps=1e-6, relu_input=True, path=_lib.PATH_FUSED)
    out, t1, kept = ops.update_forward(lib, x, z, h, bias, save_ratio=True, **kw)
    got = ops.update_backward(lib, x, z, t1, h, bias, gout, saved=kept, **kw)
    d = [t.double() for t in (x, z, h, bias, gout)]
    ro, rt1 = O.update_grouped(*d[:4], C, 1, 4, 1e-6, True)
    for a, r in zip((out, t1) + tuple(got), (ro, rt1) + tuple(O.update_backward(*d, C, 1, 4, 1e-6, True))):
        assert torch.equal(torch.isfinite(a), torch.isfinite(r))
