"""What the compiled nodes refuse: the kernels get pointers and the sizes of one tensor, so operands that
do not belong together, or lie on another device, must raise before anything is launched.  The checks come
before the nodes ask for a GPU, so most of this runs on CPU (and ``meta``) tensors."""

import pytest
import torch

import deconver_amd as dc
from deconver_amd import _lib, layers


def _t(*size, device="cpu"):
    return torch.zeros(size, device=device)


# name -> (call on the native module, part of the message)
REFUSED = {
    "few channels": (lambda n: n.linear(_t(1, 4, 8), _t(6, 5), None, 0, None, False, False), "takes 5 channels"),
    "many channels": (lambda n: n.linear(_t(1, 6, 8), _t(6, 5, 1), None, 0, None, False, False), "takes 5 channels"),
    "transposed weight": (lambda n: n.linear(_t(1, 6, 8), _t(5, 6), None, 0, None, False, True), "takes 5 channels"),
    "not three dims": (lambda n: n.linear(_t(1, 5, 8, 2), _t(6, 5), None, 0, None, False, False), "B, C, n"),
    "bias length": (lambda n: n.linear(_t(1, 5, 8), _t(6, 5), _t(5), 0, None, False, False), "bias has 5 entries"),
    "residual shape": (lambda n: n.linear(_t(1, 5, 8), _t(6, 5), None, 0, _t(1, 5, 8), False, False), "residual"),
    "residual batch": (lambda n: n.linear(_t(2, 5, 8), _t(6, 5), None, 0, _t(1, 6, 8), False, False), "residual"),
    "weight device": (lambda n: n.linear(_t(1, 5, 8), _t(6, 5, device="meta"), None, 0, None, False, False), "one device"),
    "bias device": (lambda n: n.linear(_t(1, 5, 8), _t(6, 5), _t(6, device="meta"), 0, None, False, False), "one device"),
    "residual device": (lambda n: n.linear(_t(1, 5, 8), _t(6, 5), None, 0, _t(1, 6, 8, device="meta"), False, False),
                        "one device"),
    "mlp input": (lambda n: n.mlp(_t(1, 4, 8), _t(20, 5), None, _t(5, 20), None, None), "takes 5 channels"),
    "mlp hidden": (lambda n: n.mlp(_t(1, 5, 8), _t(20, 5), None, _t(5, 16), None, None), "takes 16 channels"),
    "mlp biases": (lambda n: n.mlp(_t(1, 5, 8), _t(20, 5), _t(5), _t(5, 20), None, None), "bias has 5 entries"),
    "mlp residual": (lambda n: n.mlp(_t(1, 5, 8), _t(20, 5), None, _t(7, 20), None, _t(1, 5, 8)), "residual"),
    "mlp device": (lambda n: n.mlp(_t(1, 5, 8), _t(20, 5), None, _t(7, 20, device="meta"), None, None), "one device"),
    "update channels": (lambda n: n.projected_update(_t(1, 4, 8, 8), _t(10, 5), _t(5, 2, 3, 3), None, 5, 1, 2, 1e-8, None,
                                                     False, False, True), "takes 5 channels"),
    "update weight device": (lambda n: n.projected_update(_t(1, 5, 8, 8), _t(10, 5, device="meta"), _t(5, 2, 3, 3), None, 5,
                                                          1, 2, 1e-8, None, False, False, True), "one device"),
    "update filter device": (lambda n: n.projected_update(_t(1, 5, 8, 8), _t(10, 5), _t(5, 2, 3, 3, device="meta"), None, 5,
                                                          1, 2, 1e-8, None, False, True, True), "one device"),
    "update bias": (lambda n: n.projected_update(_t(1, 5, 8, 8), _t(10, 5), _t(5, 2, 3, 3), _t(5), 5, 1, 2, 1e-8, None,
                                                 False, False, True), "bias has 5 entries"),
    "filter table": (lambda n: n.prepare_taps(_t(1, 5, 8, 8), _t(5, 3, 3, 3), 5, 1, 2), "does not match"),
    "filter table device": (lambda n: n.prepare_taps(_t(1, 5, 8, 8), _t(5, 2, 3, 3, device="meta"), 5, 1, 2), "one device"),
    "norm weight": (lambda n: n.channel_norm(_t(1, 5, 8), _t(4), None, 1e-5), "weight has 4 entries"),
    "norm bias device": (lambda n: n.channel_norm(_t(1, 5, 8), None, _t(5, device="meta"), 1e-5), "one device"),
    "regrouping bias": (lambda n: n.regroup(_t(1, 8, 4, 8), False, _t(8)), "bias has 8 entries"),
    "regrouping layout": (lambda n: n.regroup(_t(1, 8, 8, 4).transpose(2, 3), True, None), "contiguous"),
    "columns": (lambda n: n.columns(_t(1, 2, 8, 8), [3]), "one odd extent per spatial dim"),
}


@pytest.mark.parametrize("name", REFUSED)
def test_refused_before_anything_is_launched(name):
    call, message = REFUSED[name]
    with pytest.raises((RuntimeError, ValueError), match=message):
        call(_lib.get_native())


def test_cpu_tensors_that_belong_together_are_refused_for_their_device():
    with pytest.raises(RuntimeError, match="GPU tensors only"):
        _lib.get_native().linear(_t(1, 5, 8), _t(6, 5), _t(6), 0, _t(1, 6, 8), False, False)


def _calls():
    """name -> (module on the GPU, input of the right shape, input of a wrong one)."""
    r = lambda *s: torch.rand(s, device="cuda")   # noqa: E731
    net = dict(in_channels=3, out_channels=1, spatial_dims=2, encoder_depth=(1, 1), encoder_width=(8, 16), strides=(1, 2),
               decoder_depth=(1,), kernel_size=(3, 3), groups=-1, ratio=2)
    return {
        "linear, fewer": (layers.Linear(64, 32), r(1, 64, 16, 16), r(1, 32, 16, 16)),
        "linear, more": (layers.Linear(64, 32), r(1, 64, 16, 16), r(1, 128, 16, 16)),
        "linear, streaming": (layers.Linear(64, 64), r(2, 64, 64, 1024), r(2, 32, 64, 1024)),
        "mlp": (layers.MLP(64), r(1, 64, 16, 16), r(1, 128, 16, 16)),
        "layer": (dc.Deconv(8, kernel_size=(3, 3), num_iters=2), r(1, 8, 8, 8), r(1, 16, 8, 8)),
        "downsampling": (layers.PatchConv2d(8, 16, 2, 2), r(1, 8, 16, 16), r(1, 4, 16, 16)),
        "upsampling": (layers.PatchConvTranspose2d(8, 4, 2, 2), r(1, 8, 16, 16), r(1, 4, 16, 16)),
        "stem": (layers.UnfoldConv2d(2, 8, 3, padding=1), r(1, 2, 16, 16), r(1, 3, 16, 16)),
        "network": (dc.Deconver(**net), r(1, 3, 16, 16), r(1, 4, 16, 16)),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("name", ["linear, fewer", "linear, more", "linear, streaming", "mlp", "layer", "downsampling",
                                  "upsampling", "stem", "network"])
def test_inputs_of_another_width_are_refused(name, autocast):
    module, good, bad = _calls()[name]
    module = module.cuda()
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        module(good)
        with pytest.raises((RuntimeError, ValueError)):
            module(bad)


@pytest.mark.gpu
@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("name", ["linear, fewer", "mlp", "layer", "downsampling", "upsampling", "stem", "network"])
def test_parameters_left_on_the_cpu_are_refused(name, autocast):
    module, good, _ = _calls()[name]
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast), pytest.raises((RuntimeError, ValueError)):
        module(good)


@pytest.mark.gpu
def test_residuals_and_norm_parameters_of_another_shape_or_device_are_refused():
    x = torch.rand(1, 8, 256, 256, device="cuda")
    with pytest.raises(ValueError):
        layers.Linear(8, 16).cuda()(x, residual=x)
    with pytest.raises(ValueError):
        layers.MLP(8).cuda()(x, residual=x[:, :4])
    with pytest.raises(RuntimeError):
        layers.MLP(8).cuda()(x, residual=x.cpu())
    with pytest.raises(RuntimeError):
        dc.LayerNorm(8)(x)
