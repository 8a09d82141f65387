"""Rows held in registers by one workgroup: lengths at and next to every size of workgroup and every
number of vectors a thread, whole vectors and single elements, the longest such row and the first that
takes two launches, with and without the addend, against float64.  Bounds as in the other norm tests."""

import pytest
import torch

from deconver_amd.norm import InstanceNorm2d, instance_norm

pytestmark = pytest.mark.gpu

# in 16-byte vectors; * 4 or 8 elements, and one element more (single elements from there on)
VECTORS = [1, 127, 128, 129, 512, 513, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193, 12288, 12289]


@pytest.mark.parametrize("vectors", VECTORS)
@pytest.mark.parametrize("odd", [0, 1])
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 2e-2)])
@pytest.mark.parametrize("rows", [3, 97])
def test_lengths(vectors, odd, dtype, tol, rows):
    n = vectors * (16 // dtype.itemsize) + odd
    print("case", rows, n, dtype, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = (torch.randn(1, rows, n, 1, generator=gen, device="cuda") * 3 + 20).to(dtype).requires_grad_(True)
    g, skip_g = (torch.randn(x.shape, generator=gen, device="cuda").to(dtype) for _ in range(2))
    norm = InstanceNorm2d(rows)
    y, skip = norm.with_skip(x)
    (y * g + skip * skip_g).sum().backward()
    xd = x.detach().double().requires_grad_(True)
    yd = torch.nn.functional.instance_norm(xd)
    (yd * g.double() + xd * skip_g.double()).sum().backward()
    for a, r in ((y, yd), (x.grad, xd.grad)):
        assert float((a.detach().double() - r.detach()).abs().max() / r.detach().abs().max()) < tol


# single elements, at and next to every size
@pytest.mark.parametrize("n", [127, 129, 511, 513, 1023, 1025, 2047, 2049, 4095, 4097, 8191, 8193, 12287, 12289])
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 2e-2)])
@pytest.mark.parametrize("rows", [3, 97])
def test_lengths_in_elements(n, dtype, tol, rows):
    test_lengths(n // (16 // dtype.itemsize), n % (16 // dtype.itemsize), dtype, tol, rows)


# the longest row of a few that is held, and the fewest rows from which longer ones are
@pytest.mark.parametrize("vectors", [6144, 6145, 12288])
@pytest.mark.parametrize("rows", [95, 96])
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 2e-2)])
def test_few_long_rows(vectors, rows, dtype, tol):
    test_lengths(vectors, 0, dtype, tol, rows)


def test_more_rows_than_a_launch_of_1024_threads_each_takes():
    """2^22 rows: 2^32 threads as one workgroup of 1024 a row, which is more than a launch takes."""
    rows, n = 1 << 22, 8200
    if torch.cuda.mem_get_info()[0] < 5 * rows * n:
        pytest.skip("needs 172 GB of free memory")
    x = torch.zeros(1, rows, n, dtype=torch.bfloat16, device="cuda")
    at = [0, rows // 2 + 1, rows - 1]
    x[0, at] = torch.randn(3, n, generator=torch.Generator().manual_seed(0)).to(x)
    y = instance_norm(x)
    want = torch.nn.functional.instance_norm(x[:, at].double())
    assert float((y[:, at].double() - want).abs().max() / want.abs().max()) < 2e-2
    assert float(y[0, 1].abs().max()) == 0 and float(y[0, -2].abs().max()) == 0
