"""A block as one call of the compiled nodes: the same values and gradients as its modules' calls, bit for
bit, and the modules' calls where something in it is not the stock thing."""

import copy

import pytest
import torch
from torch import nn
from torch.nn.utils import prune

import deconver_amd as dc
from deconver_amd import model as M

pytestmark = pytest.mark.gpu


def _block(nd, channels, **kw):
    torch.manual_seed(0)
    norm = {1: nn.InstanceNorm1d, 2: nn.InstanceNorm2d, 3: nn.InstanceNorm3d}[nd]
    return M.DeconverBlock(channels, norm=norm, kernel_size=(3,) * nd if nd != 2 else (5, 5), groups=kw.pop("groups", channels),
                           **kw).cuda()


def _run(block, x, autocast, one_call):
    block = copy.deepcopy(block)
    if not one_call:      # (an idle dropout is never called, but with a hook it is not the stock one)
        block.dcm.dropout.register_forward_hook(lambda *a: None)
    x = x.detach().clone().requires_grad_(True)
    with torch.autocast("cuda", torch.bfloat16, enabled=autocast):
        assert (block._one_call(x) is not None) == one_call
        y = block(x)
        with torch.no_grad():
            plain = block(x)
    y.backward(torch.randn(y.shape, generator=torch.Generator().manual_seed(1)).to(y))
    return [y, plain, x.grad] + [p.grad for p in block.parameters()]


@pytest.mark.parametrize("nd,channels,size,batch,dtype,autocast", [
    (2, 32, (20, 28), 2, torch.float32, False), (1, 8, (30,), 1, torch.float32, False), (3, 6, (5, 7, 9), 1, torch.float32, False),
    (3, 32, (8, 16, 16), 1, torch.bfloat16, False), (3, 32, (8, 12, 13), 2, torch.float32, True),
    (3, 64, (32, 32, 32), 1, torch.bfloat16, True),
    # (where no backward follows the norms fold into the projections: from rows of 98 305 voxels)
    (3, 64, (44, 48, 48), 2, torch.bfloat16, False), (3, 64, (48, 64, 32), 1, torch.bfloat16, False), (3, 64, (48, 48, 60), 1, torch.float32, True), (3, 32, (64, 40, 52), 1, torch.bfloat16, False),
    (3, 128, (52, 40, 64), 1, torch.bfloat16, False), (3, 32, (50, 46, 43), 2, torch.bfloat16, False),
    (3, 64, (48, 52, 56), 1, torch.bfloat16, True), (2, 16, (9, 11), 2, torch.bfloat16, False)])
def test_same_values(nd, channels, size, batch, dtype, autocast):
    print(nd, channels, size, batch, dtype, autocast, flush=True)
    block = _block(nd, channels)
    if dtype == torch.bfloat16 and not autocast:
        block = block.bfloat16()
        block.dcm.deconv.init.h0.data = block.dcm.deconv.init.h0.data.float()
    x = torch.randn(batch, channels, *size, generator=torch.Generator().manual_seed(2)).to("cuda", dtype)
    for a, b in zip(_run(block, x, autocast, True), _run(block, x, autocast, False)):
        assert a.dtype == b.dtype and torch.equal(a, b)


def test_what_keeps_the_modules_calls():
    x = torch.randn(1, 8, 6, 6, device="cuda")
    base = _block(2, 8)
    assert base._one_call(x) is not None

    def declined(change):
        block = copy.deepcopy(base)
        change(block)
        return block._one_call(x) is None

    class OtherLinear(dc.layers.Linear):
        pass

    def swap(b):
        b.dcm.out_proj.__class__ = OtherLinear

    def plain_bias(b):
        conv = b.mlp.block[3].linear
        bias = conv.bias.detach()
        del conv.bias
        conv.bias = bias

    for change in (lambda b: b.dcm.register_forward_hook(lambda *a: None),
                   lambda b: b.dcm.deconv.register_forward_pre_hook(lambda *a: None),
                   lambda b: b.mlp.register_full_backward_hook(lambda *a: None),
                   lambda b: b.norm2.register_forward_hook(lambda *a: None),
                   lambda b: setattr(b.dcm, "act", nn.GELU()),
                   lambda b: setattr(b.dcm.deconv, "num_iters", 2),
                   lambda b: setattr(b.dcm.deconv, "num_grad_iters", 0),
                   lambda b: setattr(b.dcm.deconv, "update_filter", True),
                   lambda b: setattr(b.mlp.block[2], "p", 0.5),
                   lambda b: setattr(b.mlp, "forward", lambda *a, **k: x),
                   lambda b: setattr(b.norm1, "affine", True),
                   lambda b: torch.nn.utils.parametrizations.weight_norm(b.mlp.block[0].linear),
                   lambda b: prune.l1_unstructured(b.mlp.block[0].linear, "bias", amount=0.5), plain_bias,
                   swap):
        assert declined(change), change
    assert base.double()._one_call(x.double()) is None and base.float()._one_call(x.cpu()) is None
    handle = nn.modules.module.register_module_forward_hook(lambda *a: None)
    try:
        assert base._one_call(x) is None
    finally:
        handle.remove()
    base.eval()
    base.mlp.block[2].p = 0.5
    assert base._one_call(x) is not None


@pytest.mark.parametrize("which", ["source", "out", "first", "second"])
def test_a_pruned_bias_is_added(which):
    block = _block(2, 8)
    bare = copy.deepcopy(block)
    parts = {"source": lambda b: b.dcm.deconv.init.linear, "out": lambda b: b.dcm.out_proj, "first": lambda b: b.mlp.block[0],
             "second": lambda b: b.mlp.block[3]}
    conv, other = parts[which](block).linear, parts[which](bare).linear
    prune.l1_unstructured(conv, "bias", amount=0.5)
    with torch.no_grad():
        other.bias.copy_(conv.bias)      # the masked values as a parameter
        x = torch.randn(1, 8, 6, 6, device="cuda")
        assert torch.equal(block(x), bare(x))
