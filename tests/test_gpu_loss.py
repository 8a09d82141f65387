"""The training loss as one node on the GPU, against its tensor operations in float64."""

import pytest
import torch
import torch.nn.functional as F

from deconver_amd import training as T

pytestmark = pytest.mark.gpu


def _oracle(logits, target):
    bce = F.binary_cross_entropy_with_logits(logits, target)
    p, y = torch.sigmoid(logits).flatten(2), target.flatten(2)
    return bce + (1 - (2 * (p * y).sum(-1) + 1) / (p.sum(-1) + y.sum(-1) + 1)).mean()


# one voxel; below, at and above a workgroup; a split with a ragged last part; more rows than the adding
# workgroup has wavefronts; the most rows; more than the node takes
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 7, 9), (1, 1, 4096), (2, 1, 65, 129), (1, 1, 8, 640, 821), (19, 1, 33, 31),
                                   (64, 16, 5), (65, 16, 5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_loss_and_gradient(shape, dtype):
    print(shape, dtype, flush=True)
    gen = torch.Generator().manual_seed(3)
    logits = (torch.randn(shape, generator=gen) * 4).to("cuda", dtype)
    target = (torch.rand(shape, generator=gen) < 0.3).float().cuda()
    x = logits.clone().requires_grad_(True)
    loss = T.dice_bce_loss(x, target)
    g, = torch.autograd.grad(loss * 3, x)
    x64 = logits.double().requires_grad_(True)
    want = _oracle(x64, target.double())
    g64, = torch.autograd.grad(want * 3, x64)
    # a thread adds up to 256 terms of one sign, then trees: 256 half units in the last place, and a few of exp's
    assert loss.dtype == torch.float32 and loss.dim() == 0
    assert abs(float(loss) - float(want)) <= 260 * 2.0 ** -24 * (abs(float(want)) + 1)
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 520 * 2.0 ** -24
    assert g.dtype == dtype
    # (the two terms of the gradient may cancel: relative to the larger of them)
    n = x64.numel()
    scale = 3 * (1.0 / n + 2.0 / (shape[0] * shape[1]))
    assert float((g.double() - g64).abs().max()) <= rel * float(g64.abs().max()) + 2.0 ** -22 * scale / n
    with torch.no_grad():
        assert torch.equal(T.dice_bce_loss(logits, target), loss.detach())


# (rows, n): a lane a row, two, four (with one idle), rows past the last trip, a wavefront a row and more parts than lanes
@pytest.mark.parametrize("shape", [(64, 16, 64), (64, 16, 5000), (100, 1, 6144), (37, 9, 8192), (5, 1, 81920), (1, 3, 160000)])
def test_parts_of_a_row(shape):
    test_loss_and_gradient(shape, torch.float32)


def test_forms_it_keeps():
    gen = torch.Generator().manual_seed(5)
    logits = torch.randn(2, 3, 10, 12, generator=gen).cuda()
    target = (torch.rand(2, 3, 10, 12, generator=gen) < 0.4).float().cuda()
    want = _oracle(logits.double(), target.double())
    close = lambda a: abs(float(a) - float(want)) < 1e-5       # noqa: E731
    x = logits.clone().requires_grad_(True)
    node = T.dice_bce_loss(x, target)
    assert type(node.grad_fn).__name__ == "_DiceBceBackward" and close(node)
    # other strides, other target types, an expanded target
    last = logits.to(memory_format=torch.channels_last).requires_grad_(True)
    a, = torch.autograd.grad(node, x, retain_graph=True)
    b, = torch.autograd.grad(T.dice_bce_loss(last, target.transpose(2, 3).contiguous().transpose(2, 3)), last)
    assert torch.equal(a, b)
    assert close(T.dice_bce_loss(x, target.to(torch.uint8))) and close(T.dice_bce_loss(x, target.double()))
    # a target that needs its gradient: tensor operations
    t = target.clone().requires_grad_(True)
    T.dice_bce_loss(x, t).backward()
    assert t.grad is not None
    # second derivatives
    d64 = logits.double().requires_grad_(True)
    g64, = torch.autograd.grad(_oracle(d64, target.double()), d64, create_graph=True)
    h64, = torch.autograd.grad(g64.square().sum(), d64)
    g, = torch.autograd.grad(node, x, create_graph=True)
    h, = torch.autograd.grad(g.square().sum(), x)
    assert float((h.double() - h64).abs().max()) <= 1e-4 * float(h64.abs().max())
    # forward mode, functorch and a recorded trace
    jvp = torch.func.jvp(lambda v: T.dice_bce_loss(v, target), (logits,), (torch.ones_like(logits),))[1]
    assert abs(float(jvp) - float(a.sum())) < 1e-5
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(logits, torch.ones_like(logits))
        assert abs(float(torch.autograd.forward_ad.unpack_dual(T.dice_bce_loss(dual, target)).tangent) - float(a.sum())) < 1e-5
    rows = torch.func.vmap(T.dice_bce_loss)(torch.stack([logits, -logits]), torch.stack([target, target]))
    assert close(rows[0])
    traced = torch.jit.trace(T.dice_bce_loss, (logits, target))
    assert abs(float(traced(-logits, target)) - float(T.dice_bce_loss(-logits, target))) < 1e-5


def test_replayed_from_a_graph():
    shape = (2, 1, 96, 96)
    x, target = torch.zeros(shape, device="cuda", requires_grad=True), torch.zeros(shape, device="cuda")
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for _ in range(2):
            torch.autograd.grad(T.dice_bce_loss(x, target), x)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        loss = T.dice_bce_loss(x, target)
        g, = torch.autograd.grad(loss, x)
    for seed in range(4):
        gen = torch.Generator().manual_seed(seed)
        with torch.no_grad():
            x.copy_(torch.randn(shape, generator=gen))
            target.copy_((torch.rand(shape, generator=gen) < 0.5).float())
        graph.replay()
        torch.cuda.synchronize()
        want = T.dice_bce_loss(x, target)
        assert torch.equal(loss, want) and torch.equal(g, torch.autograd.grad(want, x)[0])
