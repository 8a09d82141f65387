"""What a block's one call is handed, on the CPU: a recorder stands in for the compiled nodes, and an input
that says it is on the GPU for one that is.  A part whose tensors are not plain parameters keeps its
modules' calls, which read attributes."""

import pytest
import torch
from torch import nn
from torch.nn.utils import prune

from deconver_amd import _lib
from deconver_amd import model as M


class _OnGpu(torch.Tensor):
    is_cuda = property(lambda self: True)


class _Recorder:
    def __init__(self):
        self.calls = []

    def block(self, *args):
        self.calls.append(args)
        return "one call"


@pytest.fixture
def recorder(monkeypatch):
    r = _Recorder()
    monkeypatch.setattr(_lib, "get_native", lambda: r)
    return r


def _block():
    torch.manual_seed(0)
    return M.DeconverBlock(8, norm=nn.InstanceNorm2d, kernel_size=(5, 5), groups=-1, ratio=4)


def _input():
    return torch.randn(1, 8, 6, 6).as_subclass(_OnGpu)


PROJECTIONS = {"source": lambda b: b.dcm.deconv.init.linear, "out": lambda b: b.dcm.out_proj,
               "first": lambda b: b.mlp.block[0], "second": lambda b: b.mlp.block[3]}


def test_stock_block(recorder):
    block = _block()
    assert block._one_call(_input()) == "one call"
    (args,) = recorder.calls
    conv = block.mlp.block[0].linear
    assert any(a is conv.weight for a in args) and any(a is conv.bias for a in args)
    assert args[5] is None      # in_proj has no bias


@pytest.mark.parametrize("which", PROJECTIONS)
@pytest.mark.parametrize("how", ["pruned", "plain attribute"])
def test_bias_that_is_no_parameter(recorder, which, how):
    block = _block()
    conv = PROJECTIONS[which](block).linear
    if how == "pruned":
        prune.l1_unstructured(conv, "bias", amount=0.5)
    else:
        bias = conv.bias.detach().clone()
        del conv.bias
        conv.bias = bias
    assert torch.is_tensor(conv.bias) and block._one_call(_input()) is None and not recorder.calls


def test_projection_without_bias(recorder):
    block = _block()
    block.dcm.out_proj = M.Linear(32, 8, bias=False)
    assert block._one_call(_input()) == "one call"


def test_filter_that_is_no_parameter(recorder):
    block = _block()
    prune.l1_unstructured(block.dcm.deconv.init, "h0", amount=0.5)
    assert block._one_call(_input()) is None and not recorder.calls


def _replica(module):
    """A copy with its parameters as plain attributes, as nn.DataParallel's replicas have them."""
    new = module._replicate_for_data_parallel()
    for name, p in module._parameters.items():
        setattr(new, name, None if p is None else p.detach().clone())
    for name, child in module._modules.items():
        setattr(new, name, _replica(child))
    return new


def test_replica(recorder):
    assert _replica(_block())._one_call(_input()) is None and not recorder.calls


@pytest.mark.parametrize("where,name", [("", "norm1"), ("", "norm2"), ("dcm", "act")])
def test_part_that_is_no_module(recorder, where, name):
    block = _block()
    owner = block.get_submodule(where)
    delattr(owner, name)
    setattr(owner, name, lambda x: x)
    assert block._one_call(_input()) is None and not recorder.calls


ROUTE = ["fast_path_applicable", "takes_rectified_input", "context", "_fit_fast", "_regime_allows_hip", "_hip_is_ahead"]


@pytest.mark.parametrize("name", ROUTE)
@pytest.mark.parametrize("where", ["instance", "class"])
def test_replaced_method_of_the_layer(recorder, monkeypatch, where, name):
    """A method that the layer's own call would go through."""
    block = _block()
    deconv = block.dcm.deconv
    own = getattr(deconv, name)
    replacement = lambda *a, **k: own(*a, **k)      # noqa: E731
    if where == "instance":
        setattr(deconv, name, replacement)
    else:
        monkeypatch.setattr(type(deconv), name, replacement)
    assert block._one_call(_input()) is None and not recorder.calls


@pytest.mark.parametrize("name", ["norm1", "norm2"])
def test_replaced_method_of_a_norm(recorder, name):
    block = _block()
    getattr(block, name).with_skip = lambda x: (x, x)
    assert block._one_call(_input()) is None and not recorder.calls


def test_forward_only_call_that_the_library_is_ahead_on(recorder):
    """Many source channels per group: the block's call leaves the choice where the layer makes it."""
    block = M.DeconverBlock(8, norm=nn.InstanceNorm2d, kernel_size=(3, 3), groups=2, source_channels=16)
    x = _input()
    assert block._one_call(x) == "one call"
    with torch.no_grad():
        assert block._one_call(x) is None
    assert len(recorder.calls) == 1
