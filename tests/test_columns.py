"""ndc_columns: the stem's column matrix in one launch, against torch's unfold (exact: a copy)."""

import pytest
import torch

import deconver_amd as dc
from deconver_amd import _lib
from tests.helpers import hostcheck_library

# (B, C, spatial), kernel: odd and whole 16-byte rows, rows shorter than the kernel, 1-D to 3-D
CASES = [((2, 3, 11), (5,)), ((1, 2, 3, 4), (5, 5)), ((2, 3, 6, 16), (3, 3)), ((1, 2, 5, 6, 7), (3, 3, 3)),
         ((2, 1, 4, 3, 24), (3, 1, 5)), ((1, 1, 1, 1, 1), (3, 3, 3))]


def _reference(x, k):
    size = x.shape[2:]
    xp = torch.nn.functional.pad(x, [p for v in reversed(k) for p in (v // 2, v // 2)])
    for d, v in enumerate(k):
        xp = xp.unfold(2 + d, v, 1)
    n = len(k)
    return xp.permute(0, 1, *range(2 + n, 2 + 2 * n), *range(2, 2 + n)).reshape(x.shape[0], -1, size.numel())


@pytest.mark.parametrize("shape,k", CASES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_column_matrix(shape, k, dtype, device):
    x = torch.randn(shape).to(dtype).to(device)
    if device == "cuda":
        got = _lib.get_native().columns(x, list(k))
    else:
        lib = hostcheck_library()
        taps = torch.tensor(k).prod().item()
        got = torch.empty(shape[0], shape[1] * taps, x[0, 0].numel(), dtype=dtype)
        full = [1] * (3 - len(k))
        lib.columns(x.data_ptr(), got.data_ptr(), shape[0] * shape[1], *full, *shape[2:], (*full, *k),
                    _lib.NDC_BF16 if dtype == torch.bfloat16 else _lib.NDC_F32, None)
    assert torch.equal(got, _reference(x, k))


@pytest.mark.gpu
def test_an_input_that_needs_its_gradient_keeps_the_differentiable_form():
    conv = dc.layers.UnfoldConv3d(2, 16, 3, padding=1).cuda()
    x = torch.randn(1, 2, 6, 8, 10, device="cuda")
    assert torch.allclose(conv(x), conv(x.requires_grad_(True)), atol=1e-5)
    conv(x).sum().backward()
    assert x.grad is not None and x.grad.abs().sum() > 0
