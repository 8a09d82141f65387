"""The 1x1 projection as channel-first GEMMs (deconver_amd.layers.pointwise_linear) against
``conv1d`` in float64: the map the reference's ``Linear`` computes (layers/linear.py:53-58)."""

import pytest
import torch
import torch.nn.functional as F

from deconver_amd import _lib, ops
from deconver_amd.layers import Linear, pointwise_linear

pytestmark = pytest.mark.gpu


def _rel(a, ref):
    return float((a.double().cpu() - ref).abs().max() / ref.abs().max())


@pytest.mark.parametrize("B,cin,cout,n,bias", [
    (2, 32, 128, 64 * 64 * 16, True),    # many splits of the voxel axis in the weight gradient
    (1, 128, 32, 32 * 32 * 32, False),
    (3, 16, 64, 7 * 9 * 11, True),       # odd voxel count
    (2, 8, 8, 4096, True),
])
def test_pointwise_linear_matches_conv1d(B, cin, cout, n, bias):
    g = torch.Generator().manual_seed(0)
    x0 = torch.randn(B, cin, n, generator=g)
    w0 = torch.randn(cout, cin, 1, generator=g) / cin ** 0.5
    b0 = torch.randn(cout, generator=g) if bias else None
    gy0 = torch.randn(B, cout, n, generator=g)
    x = x0.cuda().bfloat16().requires_grad_(True)
    w = w0.cuda().bfloat16().requires_grad_(True)
    b = b0.cuda().requires_grad_(True) if bias else None
    y = pointwise_linear(x, w, b)
    assert y.dtype == torch.bfloat16 and y.shape == (B, cout, n) and y.is_contiguous()
    y.backward(gy0.cuda().bfloat16())
    xr = x.detach().double().cpu().requires_grad_(True)
    wr = w.detach().double().cpu().requires_grad_(True)
    br = b0.double().requires_grad_(True) if bias else None
    yr = F.conv1d(xr, wr, br)
    yr.backward(gy0.bfloat16().double())
    assert _rel(y.detach(), yr.detach()) < 1e-2
    assert _rel(x.grad, xr.grad) < 1e-2
    assert _rel(w.grad, wr.grad) < 1e-2
    if bias:
        assert b.grad.dtype == torch.float32 and _rel(b.grad, br.grad) < 1e-2


@pytest.mark.parametrize("dtype,transposed", [(torch.bfloat16, False), (torch.float32, False), (torch.bfloat16, True)])
def test_rows_beyond_the_reach_of_the_weight_gradient_kernel(dtype, transposed):
    """More than 2^24 voxels: two slices, the second one shorter and ragged."""
    n = (1 << 24) + 1001
    g = torch.Generator(device="cuda").manual_seed(1)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    x, gy = rand(1, 4, n).to(dtype), rand(1, 6, n).to(dtype)
    w = rand(*((4, 6) if transposed else (6, 4))).requires_grad_(True)
    b = rand(6).requires_grad_(True)
    pointwise_linear(x, w, b, transposed=transposed).backward(gy)
    want = gy[0].double() @ x[0].double().t()
    # (random terms: their float32 sums against the norm of the terms, sqrt(n) of about 1)
    assert float((w.grad - (want.t() if transposed else want)).abs().max()) < 4e-6 * n ** 0.5
    assert float((b.grad - gy.double().sum((0, 2))).abs().max()) < 4e-6 * n ** 0.5


def test_linear_module_under_autocast_keeps_float32_parameter_gradients():
    torch.manual_seed(0)
    lin = Linear(16, 48).cuda()
    x = torch.randn(2, 16, 8, 8, 64, device="cuda", requires_grad=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = lin(x)
    assert y.dtype == torch.bfloat16 and y.shape == (2, 48, 8, 8, 64)
    y.float().pow(2).sum().backward()
    assert lin.linear.weight.grad.dtype == torch.float32 and lin.linear.weight.grad.shape == (48, 16, 1)
    assert lin.linear.bias.grad.dtype == torch.float32 and x.grad.dtype == torch.float32
    # float32 tensors outside autocast take the same GEMM route in float32: the library
    # convolution's result to float32 rounding
    y32 = lin(x.detach())
    ref = F.conv1d(x.detach().double().flatten(2), lin.linear.weight.double(), lin.linear.bias.double()).view_as(y32)
    assert y32.dtype == torch.float32
    assert float((y32.double() - ref).abs().max() / ref.abs().max()) <= 1e-5


# (B, cin, cout, n, by the tiled GEMM): either side of each bound of the rule for bare float32 products that narrow
NARROW = [(1, 512, 256, 256, True), (1, 768, 384, 131, True), (1, 1024, 512, 64, True), (1, 1024, 512, 400, False),
          (2, 768, 60, 256, True), (2, 768, 384, 256, False), (1, 128, 64, 18310, True), (1, 128, 64, 18311, False),
          (1, 512, 256, 1144, True), (1, 512, 256, 1145, False), (1, 64, 64, 100, False), (101, 64, 32, 16, True),
          (102, 64, 32, 16, False), (59, 512, 256, 4, True), (60, 512, 256, 4, False), (70, 256, 128, 4, True),
          (1024, 128, 64, 1, False), (4, 1024, 512, 8, True), (5, 1024, 512, 8, False)]


@pytest.mark.parametrize("B,cin,cout,n,tiled", NARROW)
def test_bare_float32_products_that_narrow(B, cin, cout, n, tiled):
    g = torch.Generator(device="cuda").manual_seed(n)
    x, w = torch.randn(B, cin, n, generator=g, device="cuda"), torch.randn(cout, cin, generator=g, device="cuda") / cin ** 0.5
    y = pointwise_linear(x, w)
    assert float((y.double() - w.double() @ x.double()).norm() / y.double().norm()) < 2e-6     # float32 sums
    assert tiled or torch.equal(y, torch.bmm(w.expand(B, cout, cin), x))


# (B, cin, cout, n, by the tiled GEMM): either side of each bound of the rule for those that widen
WIDE = [(1, 16, 64, 1, True), (3, 18, 75, 77, True), (1, 64, 65, 100, True), (256, 256, 512, 1, False), (7, 512, 1024, 1, True),
        (8, 512, 1024, 1, False), (1, 256, 1024, 896, True), (1, 256, 1024, 960, False),
        (2, 128, 512, 3776, True), (2, 128, 512, 3840, False), (1, 136, 512, 3776, False)]


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("B,cin,cout,n,tiled", WIDE)
def test_bare_float32_products_that_widen(B, cin, cout, n, tiled, transposed):
    g = torch.Generator(device="cuda").manual_seed(n)
    x, w = torch.randn(B, cin, n, generator=g, device="cuda"), torch.randn(cout, cin, generator=g, device="cuda") / cin ** 0.5
    y = pointwise_linear(x, w.t().contiguous() if transposed else w, transposed=transposed)
    assert float((y.double() - w.double() @ x.double()).norm() / y.double().norm()) < 2e-6     # float32 sums
    lib = torch.bmm(w.expand(B, cout, cin), x)
    assert tiled or (y - lib).abs().max() <= 0 or transposed    # (the library has a kernel of its own for each storage)


def test_bare_float32_products_beyond_the_tiled_gemm():
    """More samples, and more output channels, than the tiled GEMM takes go by the library: forward and input gradient."""
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn((1 << 20) + 8, 32, 1, generator=g, device="cuda").requires_grad_(True)
    w = torch.randn(32, 32, generator=g, device="cuda") / 32 ** 0.5
    y = pointwise_linear(x, w)
    y.backward(x.detach())
    for got, m in ((y.detach(), w), (x.grad, w.t())):
        assert float((got - (x.detach().flatten(1) @ m.t())[..., None]).abs().max()) < 1e-4
    x, w = torch.randn(1, 1, 3, generator=g, device="cuda"), torch.randn((1 << 20) + 8, 1, generator=g, device="cuda")
    assert torch.equal(pointwise_linear(x, w), w * x)


# ... the route as well as the error: the tiled GEMM's bits, or the library's
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("B,cin,cout,n,tiled", WIDE)
def test_products_that_widen_go_by_their_rule(B, cin, cout, n, tiled, transposed):
    g = torch.Generator(device="cuda").manual_seed(n)
    x, w = torch.randn(B, cin, n, generator=g, device="cuda"), torch.randn(cout, cin, generator=g, device="cuda") / cin ** 0.5
    stored = w.t().contiguous() if transposed else w
    y = pointwise_linear(x, stored, transposed=transposed)
    if tiled:
        assert torch.equal(y, ops.gemm(_lib.get_library(), x, stored, transposed=transposed)[0])
    else:
        assert torch.equal(y, torch.bmm((stored.t() if transposed else stored).expand(B, cout, cin), x))


# (B, cin, cout, n, by the tiled GEMM): input gradients of 2 GFLOP and more whose samples fill half a tile or less, or more
@pytest.mark.parametrize("B,cin,cout,n,tiled", [(1050, 256, 256, 16, False), (525, 512, 128, 32, False), (264, 128, 512, 64, False),
                                                (260, 256, 256, 65, True), (8393, 64, 64, 32, True)])
def test_input_gradients_of_samples_of_few_voxels(B, cin, cout, n, tiled):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.empty(B, cin, n, device="cuda").requires_grad_(True)
    w = torch.randn(cout, cin, generator=g, device="cuda") / cin ** 0.5
    gy = torch.randn(B, cout, n, generator=g, device="cuda")
    pointwise_linear(x, w).backward(gy)
    if tiled:
        assert torch.equal(x.grad, ops.gemm(_lib.get_library(), gy, w, transposed=True)[0])
    else:
        assert torch.equal(x.grad, torch.bmm(w.t().expand(B, cin, cout), gy))
