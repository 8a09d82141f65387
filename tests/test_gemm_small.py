"""Small grids of the tiled GEMM (channels sliced over the wavefronts): both tile sizes, at the ends
of tiles, slices and steps, against float64 products."""

import pytest
import torch
import torch.nn.functional as F

from deconver_amd import _lib, ops

pytestmark = pytest.mark.gpu

# (B, cin, cout, n).  Up to 256 tiles of 32 rows x 64 voxels go to 16-row tiles, up to 1024 to 32-row ones
SHAPES = [(1, 8, 1, 2), (1, 16, 17, 33), (2, 40, 31, 65), (1, 2048, 512, 143), (1, 520, 48, 31), (1, 64, 256, 2049),
          (2, 1048, 160, 1601), (1, 64, 200, 3001), (3, 136, 96, 3500), (1, 8, 33, 10241)]


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-6), (torch.bfloat16, 4e-3)])   # as the other GEMM tests
@pytest.mark.parametrize("shape", SHAPES)
def test_products_and_tails(shape, dtype, tol):
    print("case", shape, dtype, flush=True)
    B, cin, cout, n = shape
    lib = _lib.get_library()
    gen = torch.Generator(device="cuda").manual_seed(cin + cout)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")   # noqa: E731
    x, res = rn(B, cin, n).to(dtype), rn(B, cout, n).to(dtype)
    w, bias = rn(cout, cin) / cin ** 0.5, rn(cout)
    z = torch.matmul(w.to(dtype).double(), x.double())
    u = z + bias.double()[:, None]
    rel = lambda a, r: float((a.double() - r).norm() / r.norm())     # noqa: E731
    y, kept = ops.gemm(lib, x, w, bias, res, "gelu", keep_z=True)
    assert rel(y, F.gelu(u) + res.double()) < tol and rel(kept, z) < tol
    y, _ = ops.gemm(lib, x, w.t().contiguous(), bias, res, transposed=True)
    assert rel(y, u + res.double()) < tol
