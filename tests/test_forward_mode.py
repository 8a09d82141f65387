"""The compiled nodes have no forward-mode rule: a dual tensor is refused, recorded or not, and never
runs without its tangent."""

import pytest
import torch
import torch.autograd.forward_ad as fwd

import deconver_amd as dc

pytestmark = pytest.mark.gpu


def _calls():
    layer = dc.Deconv(8, kernel_size=(3, 3)).cuda()
    return {
        "layer": (layer, (1, 8, 6, 8)),
        "linear": (dc.layers.Linear(8, 8).cuda(), (1, 8, 6, 8)),
        "mlp": (dc.layers.MLP(8).cuda(), (1, 8, 6, 8)),
        "norm": (dc.norm.native_norm(torch.nn.InstanceNorm2d)(8).cuda(), (1, 8, 6, 8)),
        "channel norm": (dc.LayerNorm(8).cuda(), (2, 8, 256, 256)),
        "regrouping": (dc.layers.PatchConv2d(8, 8, 2, 2).cuda(), (1, 8, 8, 8)),
        "stem": (dc.layers.UnfoldConv2d(2, 8, 3, padding=1).cuda(), (1, 2, 8, 8)),
    }


@pytest.mark.parametrize("name", ["layer", "linear", "mlp", "norm", "channel norm", "regrouping", "stem"])
@pytest.mark.parametrize("recorded", [True, False])
def test_dual_tensors_are_refused(name, recorded):
    module, shape = _calls()[name]
    module.requires_grad_(recorded)
    x = torch.rand(shape, device="cuda")
    with fwd.dual_level():
        with pytest.raises((RuntimeError, NotImplementedError)):
            module(fwd.make_dual(x, torch.ones_like(x)))
