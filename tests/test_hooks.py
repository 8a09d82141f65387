"""Modules whose work runs inside another call on the GPU are called as modules where a hook watches them
or their class is not the package's own."""

import copy

import pytest
import torch
from torch import nn

import deconver_amd as dc
from deconver_amd import layers

pytestmark = pytest.mark.gpu


def _run(module, x, autocast):
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        y = module(x)
    y.float().sum().backward()
    return y


@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("index", [0, 3])
def test_hooks_on_the_projections_of_an_mlp_fire(index, autocast):
    mlp = layers.MLP(64).cuda()
    seen, width = [], 256 if index == 0 else 64
    linear = mlp.block[index]
    linear.register_forward_pre_hook(lambda m, a: seen.append("pre"))
    linear.register_forward_hook(lambda m, a, out: seen.append(out.shape[1]))
    linear.register_full_backward_hook(lambda m, gi, go: seen.append("back"))
    _run(mlp, torch.rand(2, 64, 8, 64, device="cuda", requires_grad=True), autocast)
    assert seen == ["pre", width, "back"]


def test_hooks_on_the_parts_of_an_mlp_see_their_own_results():
    """The first projection's before the GELU, and the GELU's."""
    mlp, seen = layers.MLP(64).cuda(), {}
    for index in (0, 1, 4):
        mlp.block[index].register_forward_hook(lambda m, a, out, index=index: seen.update({index: out}))
    x = torch.randn(2, 64, 8, 64, device="cuda")
    y = mlp(x)
    first = mlp.block[0].linear
    want = torch.nn.functional.conv1d(x.double().flatten(2), first.weight.detach().double(), first.bias.detach().double())
    assert float((seen[0].detach().flatten(2) - want).norm() / want.norm()) < 1e-6      # float32 sums of 64 products
    want = torch.nn.functional.gelu(want)
    assert float((seen[1].detach().flatten(2) - want).norm() / want.norm()) < 1e-6
    assert torch.equal(seen[4], y)


def test_hooks_on_all_modules_see_the_parts_of_a_block():
    block = dc.DeconverBlock(8, kernel_size=(3, 3)).cuda()
    seen = []
    handle = nn.modules.module.register_module_forward_hook(lambda m, a, out: seen.append(m))
    try:
        _run(block, torch.rand(1, 8, 8, 8, device="cuda"), True)
    finally:
        handle.remove()
    for module in (block.norm1, block.dcm.in_proj, block.dcm.act, block.norm2, *block.mlp.block):
        assert any(m is module for m in seen), module


def test_a_projection_of_another_class_is_called():
    class Doubled(layers.Linear):
        def forward(self, x, *args, **kwargs):
            return 2 * super().forward(x, *args, **kwargs)

    mlp = layers.MLP(8).cuda()
    plain = copy.deepcopy(mlp)
    second = Doubled(32, 8).cuda()
    second.load_state_dict(mlp.block[3].state_dict())
    mlp.block[3] = second
    x = torch.rand(1, 8, 8, 8, device="cuda")
    torch.testing.assert_close(mlp(x), 2 * plain(x), rtol=1e-5, atol=1e-5)   # one float32 chain, twice


def test_a_hooked_norm_inside_the_layer_norm_is_called():
    block = dc.DeconverBlock(8, kernel_size=(3, 3)).cuda()
    seen = []
    block.norm1.norm.register_forward_hook(lambda m, a, out: seen.append(out.shape))
    _run(block, torch.rand(1, 8, 8, 8, device="cuda"), True)
    assert seen == [(1, 8, 8, 8)]


def test_a_loss_on_the_hooked_projection_of_a_mixer_reaches_its_input():
    """The hook sees the projection's own output, and gradients that reach it past the layer count:
    input and weight gradients against the same mixer in float64 on the CPU."""
    torch.manual_seed(0)
    mixer = dc.DeconvMixer(64, 64, kernel_size=(3, 3, 3), ratio=4, groups=-1)
    with torch.no_grad():
        mixer.deconv.init.linear.linear.bias.add_(1.0)
    ref = copy.deepcopy(mixer).double()
    mixer = mixer.cuda()
    x0, g0 = torch.randn(2, 64, 8, 8, 64), torch.randn(2, 64, 8, 8, 64)

    def run(module, x, g):
        kept = []
        module.in_proj.register_forward_hook(lambda m, a, out: kept.append(out))
        y = module(x)
        (y * g).sum().add((kept[0].double() ** 2).sum()).backward()
        return x.grad.double().cpu(), module.in_proj.linear.weight.grad.double().cpu()

    x = x0.cuda().bfloat16().requires_grad_(True)
    assert mixer.deconv.takes_rectified_input(x)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        got = run(mixer, x, g0.cuda().bfloat16())
    want = run(ref, x0.bfloat16().double().requires_grad_(True), g0.bfloat16().double())
    for a, b in zip(got, want):     # (bfloat16 tensors along the way: as the mixer's other test)
        assert torch.nn.functional.cosine_similarity(a.flatten(), b.flatten(), dim=0) > 0.998
