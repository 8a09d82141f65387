"""``MLP`` as one compiled node: what it gives against the same module in float64 on the CPU."""

import copy

import pytest
import torch

from deconver_amd.layers import MLP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 2e-2)])   # 2e-2: the node's bf16 chain
@pytest.mark.parametrize("out_channels", [24, 8])
@pytest.mark.parametrize("with_residual", [False, True])
def test_output_of_another_width(out_channels, with_residual, dtype, tol):
    torch.manual_seed(0)
    mlp = MLP(16, out_channels=out_channels)
    ref = copy.deepcopy(mlp).double()
    mlp = mlp.cuda()
    x0 = torch.randn(2, 16, 6, 10).to(dtype)
    r0 = torch.randn(2, out_channels, 6, 10).to(dtype) if with_residual else None
    g0 = torch.randn(2, out_channels, 6, 10).to(dtype)
    x = x0.cuda().requires_grad_(True)
    y = mlp(x, residual=r0.cuda() if with_residual else None)
    assert y.shape == g0.shape and y.dtype == dtype
    y.backward(g0.cuda())
    xr = x0.double().requires_grad_(True)
    yr = ref(xr, residual=r0.double() if with_residual else None)
    yr.backward(g0.double())
    pairs = [(y, yr), (x.grad, xr.grad)] + [(p.grad, q.grad) for p, q in zip(mlp.parameters(), ref.parameters())]
    for a, b in pairs:
        a, b = a.detach().double().cpu(), b.detach()
        assert float((a - b).norm() / b.norm()) < tol
