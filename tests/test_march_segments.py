"""The 3-D kernels (bf16 dot2; float32 and odd widths) with the march cut into segments (few workgroups otherwise): two to five
segments, ragged last ones of one to five planes, plane counts just below the first cut, rows of
whole and of partial 128-byte lines, with and without the kept ratios, against the oracle in
float64.  Bounds as in the other parity tests of bf16 and float32 storage."""

import pytest
import torch

from deconver_amd import _lib, ops
from oracle import ndc_oracle as O
from tests.helpers import host_faults, hostcheck_library, make_case

# (C, spatial, batch)
GEOMS = [(1, (11, 4, 6), 1), (1, (12, 5, 6), 2), (2, (13, 3, 10), 1), (1, (19, 9, 8), 1), (1, (33, 4, 64), 1),
         (2, (25, 10, 14), 1)]
# ... of the kernels for float32 and odd widths
PLAIN = [(1, (8, 4, 5), 1), (1, (9, 5, 6), 2), (2, (13, 3, 11), 1), (1, (17, 33, 3), 1), (1, (21, 4, 65), 1), (2, (25, 10, 1), 1)]
PLAIN_LARGE = [(64, (24, 33, 29), 1), (24, (45, 53, 77), 1), (8, (40, 38, 96), 1)]
LARGE = [(64, (32, 32, 32), 1), (24, (45, 52, 60), 1), (16, (21, 37, 192), 1)]


def _compare(lib, geom, saved, relu, device, dtype=torch.bfloat16):
    C, sp, B = geom
    x, z, h, bias, gout = make_case(C, C, 4, (3, 3, 3), sp, B=B, dtype=dtype, bias_shift=0.3,
                                    positive_z=not relu, device=device)
    kw = dict(groups=C, m=1, sc=4, eps=1e-6, relu_input=relu, path=_lib.PATH_FUSED_VECTOR)
    out, t1, *kept = ops.update_forward(lib, x, z, h, bias, save_ratio=saved, **kw)
    plain = ops.update_forward(lib, x, z, h, bias, need_t1=False, **kw)[0]
    got = ops.update_backward(lib, x, z, t1, h, bias, gout, saved=kept[0] if saved else None, **kw)
    d = [t.detach().cpu().double() for t in (x, z, h, bias, gout)]
    ro, rt1 = O.update_grouped(d[0], d[1], d[2], d[3], C, 1, 4, 1e-6, relu)
    refs = (ro, rt1) + tuple(O.update_backward(d[0], d[1], d[2], d[3], d[4], C, 1, 4, 1e-6, relu))
    errs = [O.rel_err(a.detach().cpu(), r) for a, r in zip((out, t1) + tuple(got), refs)]
    bounds = [2e-2] * 6 if dtype == torch.bfloat16 else [1e-5] * 2 + [1e-4] * 4
    assert all(e < b for e, b in zip(errs, bounds)), (geom, errs)
    assert torch.equal(out, plain)


@pytest.mark.parametrize("geom", GEOMS)
@pytest.mark.parametrize("saved", [False, True])
@pytest.mark.parametrize("relu", [False, True])
def test_segments_on_the_host_build(geom, saved, relu):
    lib = hostcheck_library()
    host_faults(lib)
    _compare(lib, geom, saved, relu, "cpu")
    n, first = host_faults(lib)
    assert n == 0, f"faults: {n} ({first})"


@pytest.mark.gpu
@pytest.mark.parametrize("geom", GEOMS + LARGE)
@pytest.mark.parametrize("saved", [False, True])
def test_segments_on_the_gpu(geom, saved):
    print("case", geom, saved, flush=True)
    _compare(_lib.get_library(), geom, saved, True, "cuda")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("geom", PLAIN)
@pytest.mark.parametrize("saved", [False, True])
def test_plain_segments_on_the_host_build(geom, saved, dtype):
    lib = hostcheck_library()
    host_faults(lib)
    _compare(lib, geom, saved, True, "cpu", dtype)
    n, first = host_faults(lib)
    assert n == 0, f"faults: {n} ({first})"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("geom", PLAIN + PLAIN_LARGE)
@pytest.mark.parametrize("saved", [False, True])
def test_plain_segments_on_the_gpu(geom, saved, dtype):
    print("case", geom, saved, dtype, flush=True)
    _compare(_lib.get_library(), geom, saved, True, "cuda", dtype)
