"""The optimiser's kernel against the library's AdamW in float64."""

import copy

import pytest
import torch
from torch import nn

from deconver_amd import training as T

pytestmark = pytest.mark.gpu


class _Bag(nn.Module):
    def __init__(self, sizes, seed=0):
        super().__init__()
        gen = torch.Generator().manual_seed(seed)
        self.p = nn.ParameterList([nn.Parameter(torch.randn(s, generator=gen)) for s in sizes])


def _grads(bag, seed, skip=()):
    gen = torch.Generator().manual_seed(100 + seed)
    for i, p in enumerate(bag.p):
        g = torch.randn(p.shape, generator=gen) * 10.0 ** (i % 7 - 3)
        p.grad = None if i in skip else g.to(p)


# one element; below, at and above a workgroup's share, with a cut vector; more tensors than one launch names;
# more than one launch of counters
SIZES = {"one": [(1,)], "edges": [(4095,), (4096,), (4097,), (3, 5, 7), (0,), (2, 8192)],
         "many": [(i % 37 + 1,) for i in range(130)], "counters": [(2,)] * 450}


@pytest.mark.parametrize("sizes", SIZES)
def test_steps(sizes):
    print(sizes, flush=True)
    bag = _Bag(SIZES[sizes]).cuda()
    ref = copy.deepcopy(bag).cpu().double()
    opt = T.make_optimizer(bag)
    want = torch.optim.AdamW(ref.parameters(), lr=1e-3, weight_decay=1e-2)
    assert isinstance(opt, torch.optim.AdamW)
    for step in range(5):
        skip = (0,) if step == 2 and len(bag.p) > 1 else ()
        _grads(bag, step, skip), _grads(ref, step, skip)
        if step == 0:      # (the first step makes the state)
            assert not opt._kernel_step()
        before = [p._version for p in bag.p]
        opt.step(), want.step()
        assert step == 0 or all(p._version > b for i, (p, b) in enumerate(zip(bag.p, before)) if i not in skip)
        if step == 1:      # what was saved goes on where it was
            opt.load_state_dict(copy.deepcopy(opt.state_dict()))
    for i, (p, q) in enumerate(zip(bag.p, ref.parameters())):
        s, r = opt.state[p], want.state[q]
        assert float(s["step"]) == float(r["step"])
        # five steps of at most four roundings each on values of either sign, and steps of about lr
        scale = lambda t: float(t.abs().max()) if t.numel() else 0.0      # noqa: E731
        assert scale(s["exp_avg"].cpu().double() - r["exp_avg"]) <= 20 * 2.0 ** -24 * 10.0 ** (i % 7 - 3) * 5
        assert scale(s["exp_avg_sq"].cpu().double() - r["exp_avg_sq"]) <= 20 * 2.0 ** -24 * scale(r["exp_avg_sq"])
        assert scale(p.detach().cpu().double() - q.detach()) <= 20 * 2.0 ** -24 * (scale(q.detach()) + 1)


@pytest.mark.parametrize("offset", [1, 2, 3])
@pytest.mark.parametrize("which", ["param", "grad"])
def test_views_of_a_flat_buffer(offset, which):
    """Parameters or gradients that no 16-byte access takes: element by element from the first on, with less
    than a workgroup's share, exactly one, and one and a part."""
    sizes = [(4095,), (4096,), (4097,), (33, 300), (1,)]
    flat = torch.empty(offset + sum(torch.Size(s).numel() for s in sizes) + 4 * len(sizes), device="cuda")
    views, at = [], offset
    for s in sizes:
        n = torch.Size(s).numel()
        views.append(flat[at:at + n].view(s))
        at += (n + 3) // 4 * 4        # (all as far from 16 bytes as the first)
    assert all(v.data_ptr() % 16 == 4 * offset for v in views)
    bag = _Bag(sizes).cuda()
    ref = copy.deepcopy(bag).cpu().double()
    if which == "param":
        for p, v in zip(bag.p, views):
            v.copy_(p.detach())
            p.data = v
    opt = T.make_optimizer(bag)
    want = torch.optim.AdamW(ref.parameters(), lr=1e-3, weight_decay=1e-2)
    for step in range(5):
        _grads(bag, step), _grads(ref, step)
        if which == "grad":
            for p, v in zip(bag.p, views):
                p.grad = v.copy_(p.grad)
        if step:
            assert opt._kernel_step()
        else:
            opt.step()
        want.step()
    for i, (p, q) in enumerate(zip(bag.p, ref.parameters())):
        s, r = opt.state[p], want.state[q]
        assert float(s["step"]) == float(r["step"])
        # as in test_steps
        scale = lambda t: float(t.abs().max())      # noqa: E731
        assert scale(s["exp_avg"].cpu().double() - r["exp_avg"]) <= 20 * 2.0 ** -24 * 10.0 ** (i % 7 - 3) * 5
        assert scale(s["exp_avg_sq"].cpu().double() - r["exp_avg_sq"]) <= 20 * 2.0 ** -24 * scale(r["exp_avg_sq"])
        assert scale(p.detach().cpu().double() - q.detach()) <= 20 * 2.0 ** -24 * (scale(q.detach()) + 1)


def test_what_the_base_class_does():
    """Forms the kernel declines, and hooks, run once."""
    count = []
    for change in ({}, {"amsgrad": True}, {"maximize": True}, {"lr": torch.tensor(1e-3)}):
        bag = _Bag([(33,), (4,)]).cuda()
        twin = copy.deepcopy(bag)
        opt = T.make_optimizer(bag, capturable=True)
        want = torch.optim.AdamW(twin.parameters(), lr=1e-3, weight_decay=1e-2, fused=True, capturable=True)
        for o in (opt, want):
            o.param_groups[0].update({k: v.cuda() if torch.is_tensor(v) else v for k, v in change.items()})
        opt.register_step_post_hook(lambda *a: count.append(1))
        for step in range(3):
            _grads(bag, step), _grads(twin, step)
            opt.step(), want.step()
        assert len(count) == 3
        count.clear()
        for p, q in zip(bag.p, twin.p):
            assert torch.allclose(p, q, rtol=1e-6, atol=1e-6)
    # gradients of another layout than their parameter: refused there
    bag = nn.ParameterList([nn.Parameter(torch.ones(4, 6, device="cuda"))])
    opt = T.AdamW(bag, fused=True)
    bag[0].grad = torch.ones(4, 6, device="cuda")
    opt.step()
    bag[0].grad = torch.ones(6, 4, device="cuda").t()
    assert not opt._kernel_step()
    with pytest.raises(RuntimeError):
        opt.step()
    bag[0].grad = torch.ones(4, 6, device="cuda")
    # a closure
    assert float(opt.step(lambda: torch.tensor(3.0))) == 3.0


def test_recorded():
    bag = _Bag([(5000,), (7,)]).cuda()
    twin = copy.deepcopy(bag)
    opt, want = T.make_optimizer(bag, capturable=True), T.make_optimizer(twin, capturable=True)
    _grads(bag, 0), _grads(twin, 0)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        opt.step(), want.step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        opt.step()
    for seed in range(1, 5):
        for p, q in zip(bag.p, twin.p):
            g = torch.randn(p.shape, generator=torch.Generator().manual_seed(seed)).cuda()
            p.grad.copy_(g), q.grad.copy_(g)
        graph.replay()
        torch.cuda.synchronize()
        want.step()
        for p, q in zip(bag.p, twin.p):
            assert torch.equal(p, q) and torch.equal(opt.state[p]["step"], want.state[q]["step"])
