"""The channel norm's register-held kernels at the edges of what they hold: channel counts around
the slices and the register blocks, rows that fill no run of lanes, several workgroups a sample and
the count from which the two-loop kernels serve; and a block's one-pass form against the module's."""

import pytest
import torch

import deconver_amd as dc
from deconver_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 3, 65), (2, 7, 130), (1, 9, 127), (3, 33, 257), (1, 64, 4098), (2, 129, 511),
                                   (1, 256, 1000), (1, 257, 1000), (1, 8, 300002)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shift", [0, 1])       # 1: buffers aligned to one element only
def test_kernels_against_float64(shape, dtype, shift):
    print("case", shape, dtype, shift, flush=True)
    B, C, n = shape
    gen = torch.Generator(device="cuda").manual_seed(sum(shape))

    def rand():
        t = torch.empty(B * C * n + shift, device="cuda", dtype=dtype)
        return t[shift:].copy_(torch.randn(B * C * n, device="cuda", generator=gen)).view(B, C, n)

    x, gy = rand().add_(3.0), rand()
    w, b = torch.rand(C, device="cuda", generator=gen) + 0.5, torch.randn(C, device="cuda", generator=gen)
    lib = _lib.get_library()
    y, stats = ops.chnorm_forward(lib, x, w, b, 1e-5)
    gx, gw, gb = ops.chnorm_backward(lib, gy, x, stats, w)
    xd, wd, bd = x.double().requires_grad_(True), w.double().requires_grad_(True), b.double().requires_grad_(True)
    ref = torch.nn.functional.layer_norm(xd.movedim(1, -1), (C,), wd, bd, 1e-5).movedim(-1, 1)
    want = torch.autograd.grad(ref, (xd, wd, bd), gy.double())
    # one rounding to the stored type (2^-24, 2^-9) on values of the norm's size, a few in the sums; from
    # three channels on (with one or two the true input gradient is zero or nearly so)
    tol = 2e-6 if dtype == torch.float32 else 4e-3
    err = lambda a, r: float((a.double() - r).norm().detach() / r.detach().norm())  # noqa: E731
    assert err(y, ref) < tol
    for got, r in zip((gx, gw, gb), want):
        assert err(got, r) < tol


def test_a_block_gets_the_bits_of_the_three_pass_form():
    """bfloat16 values under bfloat16 autocast: normalised and rounded in one pass, forward and
    backward, against float32 normalisation between two conversions."""
    torch.manual_seed(3)
    norm = dc.LayerNorm(64).cuda()
    with torch.no_grad():
        norm.norm.weight.uniform_(0.5, 1.5)
        norm.norm.bias.uniform_(-0.5, 0.5)
    consumer = dc.layers.Linear(64, 64).cuda()
    g = torch.randn(2, 64, 40, 50, 20, device="cuda").bfloat16()
    x = torch.randn_like(g).requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        one, three = norm.for_projection(x, consumer), norm(x)
    assert one.dtype == torch.bfloat16 and three.dtype == torch.float32
    assert torch.equal(one, three.bfloat16())
    assert torch.equal(*(torch.autograd.grad(y, x, g)[0] for y in (one, three.bfloat16())))
    seen = []
    handle = norm.register_forward_hook(lambda m, a, out: seen.append(out.dtype))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert norm.for_projection(x, consumer).dtype == torch.float32 and seen == [torch.float32]
    handle.remove()
