"""Saved-tensor hooks around the compiled nodes: what they give back is looked at before a kernel reads it."""

import pytest
import torch
from torch import nn

import deconver_amd as dc
from deconver_amd import _lib, layers

pytestmark = pytest.mark.gpu

MODULES = {
    "linear": (lambda: layers.Linear(8, 12), (2, 8, 16, 16)),
    "mlp": (lambda: layers.MLP(8), (2, 8, 16, 16)),
    "layer": (lambda: dc.Deconv(8, kernel_size=(3, 3)), (2, 8, 16, 16)),
    "layer, two updates": (lambda: dc.Deconv(8, kernel_size=(3, 3, 3), num_iters=2), (2, 8, 8, 8, 8)),
    "instance norm": (lambda: dc.norm.InstanceNorm2d(8), (2, 8, 16, 16)),
    "channel norm": (lambda: dc.LayerNorm(8), (2, 8, 128, 128)),
}


def _gradients(name, autocast, pack=lambda t: t, unpack=lambda t: t):
    torch.manual_seed(0)
    build, shape = MODULES[name]
    module = build().cuda()
    x = torch.rand(shape, device="cuda", requires_grad=True)
    with torch.autograd.graph.saved_tensors_hooks(pack, unpack), torch.autocast("cuda", torch.bfloat16, enabled=autocast):
        y = module(x)
    y.float().sum().backward()
    return [x.grad] + [p.grad for p in module.parameters()]


def _spread(t):
    """The same values with strides of another layout."""
    return torch.stack([t, t], dim=-1)[..., 0] if t.dim() in (3, 4, 5) and t.is_floating_point() else t


@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("name", ["linear", "mlp", "instance norm", "channel norm"])
def test_tensors_that_come_back_in_another_layout(name, autocast):
    for a, b in zip(_gradients(name, autocast, unpack=_spread), _gradients(name, autocast)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("name", MODULES)
@pytest.mark.parametrize("unpack", [lambda t: t.to(torch.float16) if t.is_floating_point() else t, lambda t: t[:1],
                                    lambda t: t.cpu()], ids=["type", "shape", "device"])
def test_tensors_that_come_back_as_others_are_refused(unpack, name, autocast):
    with pytest.raises((RuntimeError, ValueError, TypeError)):
        _gradients(name, autocast, unpack=unpack)


@pytest.mark.parametrize("name", MODULES)
def test_tensors_kept_on_the_cpu(name):
    for a, b in zip(_gradients(name, True, lambda t: t.cpu(), lambda t: t.cuda()), _gradients(name, True)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("hidden,cin", [(96, 32), (160, 32), (256, 64), (128, 64)])
def test_weights_of_another_width_are_refused_by_the_mlp_on_chip(hidden, cin):
    """Two weights that fit each other and the kept input, but not the widths the kernels are built for."""
    gen = torch.Generator(device="cuda").manual_seed(0)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda")   # noqa: E731
    x, w1, w2 = rand(1, 32, 4096).bfloat16(), rand(128, 32), rand(32, 128)
    other = {(1, 32, 4096): rand(1, cin, 4096).bfloat16(), (128, 32): rand(hidden, cin), (32, 128): rand(32, hidden)}
    x, w1, w2 = (t.requires_grad_(True) for t in (x, w1, w2))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: other[tuple(t.shape)]):
        y = _lib.get_native().mlp(x, w1, None, w2, None, None)
    with pytest.raises(ValueError, match="saved weights came back"):
        y.backward(torch.ones_like(y))
