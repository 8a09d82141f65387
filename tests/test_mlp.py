"""``MLP`` as one compiled node: what it gives against the same module in float64 on the CPU."""

import copy

import pytest
import torch

from deconver_amd import _lib
from deconver_amd.layers import MLP, pointwise_linear

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


def _bias_grad_reference(z, b, gz):
    """float64 sums of gz * gelu'(z + b), each row over batch and voxels, and their terms' norms."""
    u = (z.double() + b.double()[:, None]).requires_grad_(True)
    torch.nn.functional.gelu(u).backward(gz.double())
    return u.grad.sum((0, 2)), u.grad.norm(dim=(0, 2))


# by what makes the gradient of the hidden tensor: the kernel that keeps it on chip; the streaming GEMM; the tiled one, its channels sliced over the
# wavefronts (both tile sizes), in whole and in ragged tiles; the library's and a pass
ROUTES = [(2, 64, 256, 65536), (2, 128, 512, 65536), (1, 64, 256, 1000), (1, 64, 256, 4099), (1, 64, 256, 20001), (2, 30, 120, 777),
          (1, 256, 1024, 8192)]


@pytest.mark.parametrize("B,c,hidden,n", ROUTES)
def test_bias_gradient_behind_the_gelu_is_not_rounded(B, c, hidden, n):
    """bfloat16, with weights that pick one channel each, so that the hidden tensor and its gradient's
    product are exact: what is left is the activation's derivative (3e-7) and float32 sums.  Terms
    rounded to bfloat16 would put 1e-3 of their norm into the result."""
    gen = torch.Generator(device="cuda").manual_seed(n)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")   # noqa: E731
    mlp = MLP(c, hidden_channels=hidden).cuda()
    first, second = mlp.block[0].linear, mlp.block[3].linear
    unit = torch.arange(hidden, device="cuda")
    with torch.no_grad():
        first.weight.zero_()[unit, unit % c, 0] = 0.5
        second.weight.zero_()[(unit * 7) % c, unit, 0] = 2.0
    x, g = rand(B, c, n).bfloat16(), rand(B, c, n).bfloat16()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = mlp(x.requires_grad_(True))
    y.backward(g)
    want, norm = _bias_grad_reference(0.5 * x.detach().float()[:, unit % c], first.bias.detach(), 2.0 * g.float()[:, (unit * 7) % c])
    assert float(((first.bias.grad - want).abs() / norm).max()) < 2e-5


def test_bias_gradient_of_a_projection_with_its_gelu_is_not_rounded():
    torch.manual_seed(0)
    x = torch.randn(2, 16, 4000, device="cuda").bfloat16()
    w = torch.zeros(48, 16, device="cuda")
    w[torch.arange(48), torch.arange(48) % 16] = 0.5
    b = torch.randn(48, device="cuda", requires_grad=True)
    g = torch.randn(2, 48, 4000, device="cuda").bfloat16()
    pointwise_linear(x, w, b, act="gelu").backward(g)
    want, norm = _bias_grad_reference(0.5 * x.float().repeat(1, 3, 1), b.detach(), g)
    assert float(((b.grad - want).abs() / norm).max()) < 2e-5


def _float64_mlp(x, w1, b1, w2, b2, res, g):
    """Value and gradients in float64 of the operands as bfloat16 holds them (weights rounded, as the
    products take them)."""
    leaves = [t.detach().double().requires_grad_(True) if t is not None else None
              for t in (x, w1.bfloat16(), b1, w2.bfloat16(), b2, res)]
    xd, w1d, b1d, w2d, b2d, rd = leaves
    u = w1d @ xd if b1d is None else w1d @ xd + b1d[:, None]
    y = w2d @ torch.nn.functional.gelu(u)
    if b2d is not None:
        y = y + b2d[:, None]
    if rd is not None:
        y = y + rd
    y.backward(g.double())
    return y.detach(), [t.grad if t is not None else None for t in leaves]


# the size the hidden tensor stays on chip from, with 64 and 32 channels; tiles that fill the workgroups of
# the backward and each workgroup size of the forward evenly, and one over
@pytest.mark.parametrize("B,c,n", [(1, 64, 32768), (1, 64, 65600), (1, 64, 131072), (3, 64, 43712), (1, 64, 262208), (1, 32, 4096),
                                   (2, 32, 65600), (1, 32, 196608)])
@pytest.mark.parametrize("bias,residual,wdtype", [(True, True, torch.float32), (False, False, torch.bfloat16)])
def test_hidden_tensor_on_chip(B, c, n, bias, residual, wdtype):
    """Bounds: the result and gx carry one rounding (2^-9) of themselves and of the hidden values they
    sum (their errors independent, so no more in norm); the weight gradients the hidden roundings only;
    the bias gradients float32 sums and the derivative's 3e-7."""
    gen = torch.Generator(device="cuda").manual_seed(c + n)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")   # noqa: E731
    x, g = rand(B, c, n).bfloat16(), rand(B, c, n).bfloat16()
    w1, w2 = (rand(4 * c, c) / c ** 0.5).to(wdtype), (rand(c, 4 * c) / (4 * c) ** 0.5).to(wdtype)
    b1, b2 = (rand(4 * c), rand(c)) if bias else (None, None)
    res = rand(B, c, n).bfloat16() if residual else None
    leaves = [t.requires_grad_(True) if t is not None else None for t in (x, w1, b1, w2, b2, res)]
    native = _lib.get_native()
    y = native.mlp(*leaves)
    y.backward(g)
    with torch.no_grad():
        assert torch.equal(native.mlp(*leaves), y)
    want, grads = _float64_mlp(x, w1, b1, w2, b2, res, g)
    err = lambda a, b: float((a.double() - b).norm() / b.norm())   # noqa: E731
    assert err(y.detach(), want) < 4e-3
    for t, ref, tol in zip(leaves, grads, (4e-3, 6e-3, 2e-5, 6e-3, 2e-5, 1e-6)):
        if t is not None and t.dtype == torch.bfloat16:
            tol = max(tol, 4e-3)
        assert t is None or err(t.grad, ref) < tol, (tuple(t.shape), err(t.grad, ref))


# 32 channels: the tiles that two wavefronts share (an odd number of them, the most) and one more
@pytest.mark.parametrize("B,n", [(1, 4160), (3, 4160), (1, 32768), (1, 32832)])
@pytest.mark.parametrize("bias,residual,wdtype", [(True, True, torch.float32), (False, False, torch.bfloat16)])
def test_tiles_of_two_wavefronts(B, n, bias, residual, wdtype):
    test_hidden_tensor_on_chip(B, 32, n, bias, residual, wdtype)


@pytest.mark.parametrize("c,n", [(32, 4096 + 64), (64, 32768)])
def test_some_of_the_gradients(c, n):
    """Where only some are asked for they are the same as among all."""
    gen = torch.Generator(device="cuda").manual_seed(c)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")   # noqa: E731
    leaves = [t.requires_grad_(True) for t in (rand(1, c, n).bfloat16(), rand(4 * c, c) / c ** 0.5, rand(4 * c), rand(c, 4 * c) / c, rand(c))]
    g = rand(1, c, n).bfloat16()
    y = _lib.get_native().mlp(*leaves, None)
    want = torch.autograd.grad(y, leaves, g, retain_graph=True)
    for some in ((0,), (3,), (4,), (3, 4), (1,), (2,), (1, 2, 3, 4), (0, 1, 2), (0, 4), (0, 3), (1, 3)):
        print("case", c, some, flush=True)
        for i, a in zip(some, torch.autograd.grad(y, [leaves[i] for i in some], g, retain_graph=True)):
            assert torch.equal(a, want[i]), (some, i)


@pytest.mark.parametrize("frozen", ["x", "w1", "w2"])
def test_partly_frozen_mlp_gives_the_same_gradients(frozen):
    gen = torch.Generator(device="cuda").manual_seed(1)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")   # noqa: E731
    ops_ = dict(x=rand(1, 32, 131072).bfloat16(), w1=rand(128, 32) / 6, w2=rand(32, 128) / 11)
    g = rand(1, 32, 131072).bfloat16()
    got = []
    for keep in (True, False):
        t = {k: v.clone().requires_grad_(keep or k != frozen) for k, v in ops_.items()}
        _lib.get_native().mlp(t["x"], t["w1"], None, t["w2"], None, None).backward(g)
        got.append(t)
    for k in ops_:
        if k == frozen:
            assert got[1][k].grad is None
        else:
            a, b = got[0][k].grad.double(), got[1][k].grad.double()
            assert float((a - b).norm() / a.norm()) < 1e-2


@pytest.mark.parametrize("c,n", [(32, 4096), (64, 32768)])
def test_weights_at_an_odd_element(c, n):
    """bfloat16 weights that are views one element into a flat buffer: the same bits as aligned ones."""
    gen = torch.Generator(device="cuda").manual_seed(c)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")   # noqa: E731
    x, g = rand(1, c, n).bfloat16(), rand(1, c, n).bfloat16()
    flat = rand(8 * c * c + 2).bfloat16() / c ** 0.5
    odd = [flat[1:1 + 4 * c * c].view(4 * c, c), flat[1 + 4 * c * c:1 + 8 * c * c].view(c, 4 * c)]
    assert all(w.data_ptr() % 4 == 2 for w in odd)
    got = []
    for weights in (odd, [w.clone() for w in odd]):
        leaves = [t.detach().requires_grad_(True) for t in (x, *weights)]
        y = _lib.get_native().mlp(leaves[0], leaves[1], None, leaves[2], None, None)
        y.backward(g)
        got.append([y] + [t.grad for t in leaves])
    for a, b in zip(*got):
        assert torch.equal(a, b)
