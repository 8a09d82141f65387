"""The tiled GEMMs of the projections (ndc_gemm: forward and input gradient with their tails;
ndc_weight_grad: weight and bias gradient in one pass) against float64 products of the same
operands, at the sizes where tiles, stages and splits have ends."""

import pytest
import torch
import torch.nn.functional as F

from deconver_amd import _lib, ops
from tests.helpers import hostcheck_library

# (B, cin, cout, n): one element; a voxel past a tile; ragged depth and rows; tiny grids over many
# channels (channels sliced over the wavefronts); an odd row length; a tile of one voxel pair
SHAPES = [(1, 1, 1, 1), (2, 64, 32, 129), (3, 130, 70, 77), (1, 54, 64, 1000), (2, 1048, 96, 105), (1, 64, 33, 4099),
          (2, 8, 40, 2), (1, 512, 160, 64)]
DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]
DTYPES = [(torch.float32, 2e-6), (torch.bfloat16, 4e-3)]


def _setup(device, shape, dtype):
    lib = hostcheck_library() if device == "cpu" else _lib.get_library()
    B, cin, cout, n = shape
    gen = torch.Generator().manual_seed(cin + cout)
    rn = lambda *s: torch.randn(*s, generator=gen)   # noqa: E731
    x, res, mask, g = rn(B, cin, n), rn(B, cout, n), rn(B, cout, n), rn(B, cout, n)
    w, bias = rn(cout, cin) / cin ** 0.5, rn(cout)
    return lib, [t.to(device=device, dtype=dtype) for t in (x, res, mask, g)], w.to(device), bias.to(device)


def _rel(a, ref):
    ref = ref.double()
    return float((a.double() - ref).norm() / ref.norm().clamp_min(1e-30))


@pytest.mark.parametrize("dtype,tol", DTYPES)
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("device", DEVICES)
def test_products_with_their_tails(device, shape, dtype, tol):
    lib, (x, res, mask, _), w, bias = _setup(device, shape, dtype)
    wt = w.t().contiguous()
    z = torch.matmul(w.to(dtype).double(), x.double())
    u = z + bias.double()[:, None]
    y, _ = ops.gemm(lib, x, w)
    assert _rel(y, z) < tol
    y, zk = ops.gemm(lib, x, w, bias, res, "gelu", keep_z=True)
    assert _rel(y, F.gelu(u) + res.double()) < tol and _rel(zk, z) < tol
    y, _ = ops.gemm(lib, x, w, bias, None, "relu")
    assert _rel(y, u.clamp_min(0)) < tol
    y, _ = ops.gemm(lib, x, wt, bias, res, mask=mask, transposed=True)
    assert _rel(y, torch.where(mask.double() > 0, u + res.double(), 0.0)) < tol
    v = (res.double() + bias.double()[:, None]).requires_grad_(True)
    F.gelu(v).sum().backward()
    y, _ = ops.gemm(lib, x, wt, bias, res, "gelu_grad", transposed=True)
    assert _rel(y, z * v.grad) < tol


@pytest.mark.parametrize("dtype,tol", DTYPES)
@pytest.mark.parametrize("shape", SHAPES + [(1, 32, 256, 3000), (2, 300, 48, 2100), (2, 96, 128, 1537)])
@pytest.mark.parametrize("device", DEVICES)
def test_weight_and_bias_gradient(device, shape, dtype, tol):
    lib, (x, _, _, g), _, _ = _setup(device, shape, dtype)
    gw, gb = ops.weight_grad(lib, g, x, need_bias_grad=True)
    assert _rel(gw, torch.matmul(g.double(), x.double().transpose(1, 2)).sum(0)) < 4e-6
    assert _rel(gb, g.double().sum((0, 2))) < 4e-6
    again, none = ops.weight_grad(lib, g, x)
    assert torch.equal(again, gw) and none is None


# voxel tiles of 128 (the last two for a ragged depth and a last tile of one voxel), 64 and 32
@pytest.mark.parametrize("dtype,tol", DTYPES)
@pytest.mark.parametrize("shape", SHAPES + [(1, 64, 256, 4099), (2, 64, 96, 30001), (3, 30, 120, 257)])
@pytest.mark.parametrize("device", DEVICES)
def test_gelu_gradient_with_its_sums(device, shape, dtype, tol):
    """The sums are of the float32 values: a rounding to bfloat16 in their terms would show as 1e-3."""
    if device == "cpu" and shape[3] > 5000:
        pytest.skip("the host build's loops")
    lib, (x, res, _, _), w, bias = _setup(device, shape, dtype)
    z = torch.matmul(w.to(dtype).double(), x.double())
    v = (res.double() + bias.double()[:, None]).requires_grad_(True)
    F.gelu(v).sum().backward()
    gz, gb = ops.gemm_gelu_grad(lib, x, w.t().contiguous(), res, bias)
    want = z * v.grad
    assert _rel(gz, want) < tol
    # per term: the product's float32 sums and the derivative's 3e-7; over the terms as their norm grows
    assert float((gb.double() - want.sum((0, 2))).abs().max()) < 4e-6 * float(want.norm(dim=(0, 2)).max()) + 1e-6


@pytest.mark.parametrize("rows,cols", [(1, 1), (7, 33), (2048, 5), (2049, 40), (4096, 96)])
@pytest.mark.parametrize("device", DEVICES)
def test_column_sums(device, rows, cols):
    lib = hostcheck_library() if device == "cpu" else _lib.get_library()
    part = torch.randn(rows, cols, generator=torch.Generator().manual_seed(rows)).to(device)
    want = part.double().sum(0)
    assert float((ops.column_sums(lib, part) - want).abs().max()) < 2e-6 * max(1.0, rows ** 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(256, 64), (64, 54)])
def test_weight_gradient_over_long_rows(rows, cols):
    """Rows long enough for the deep stages, with a ragged end."""
    lib, n = _lib.get_library(), (1 << 19) + 21
    torch.manual_seed(0)
    g, x = (torch.randn(1, c, n, device="cuda").bfloat16() for c in (rows, cols))
    gw, gb = ops.weight_grad(lib, g, x, need_bias_grad=True)
    assert _rel(gw, g[0].double() @ x[0].double().t()) < 1e-5 and _rel(gb, g.double().sum((0, 2))) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("cin,cout,n", [(64, 256, 1280), (128, 512, 1000), (320, 64, 5000)])
def test_small_grids_keep_one_order_of_sums(cin, cout, n):
    """bf16 grids of 129 to 256 tiles of 32 x 64 add their channels in the order of smaller ones: bit-equal columns.
    (Channels of very different sizes, so that another order rounds otherwise.)"""
    assert 128 < -(-n // 64) * -(-cout // 32) <= 256
    lib, (x, _, _, _), w, _ = _setup("cuda", (1, cin, cout, n), torch.bfloat16)
    x *= torch.logspace(-3, 3, cin, device="cuda").roll(cin // 2)[:, None]
    half = n // 256 * 128
    assert torch.equal(ops.gemm(lib, x, w)[0][..., :half], ops.gemm(lib, x[..., :half].contiguous(), w)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("B,cin,cout,n", [(96, 1024, 256, 16), (180, 512, 128, 64), (24, 1024, 256, 16), (40, 256, 128, 32)])
def test_small_float32_grids_of_few_voxels_are_sliced(B, cin, cout, n):
    """601 to 1024 of the larger tiles over samples of at most 64 voxels, 129 to 256 over at most 32: the bits of fewer samples."""
    lib, (x, _, _, _), w, _ = _setup("cuda", (B, cin, cout, n), torch.float32)
    few = max(1, 100 // (cout // 32)) if B * cout // 32 <= 256 else B // 2
    assert torch.equal(ops.gemm(lib, x, w)[0][:few], ops.gemm(lib, x[:few].contiguous(), w)[0])


# rows of 32 and 64 a workgroup, one chain of sums and several; ragged channels, rows and voxels
PARTS = [(1, 33, 40, 38501), (2, 100, 130, 9001), (1, 32, 64, 52001), (2, 72, 30, 20003), (1, 1030, 96, 13000)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", PARTS)
def test_float32_products_of_parts(shape):
    """float32 products made of bf16 parts, over grids that are not sliced.  The error of a chain of 64 channels is
    1.1e-7 of the result's norm, that of chains of 32 and their sum 0.7e-7 .. 1.4e-7; the values' mean is off by noise."""
    print("case", shape, flush=True)
    lib, (x, res, _, g), w, bias = _setup("cuda", shape, torch.float32)
    z = torch.matmul(w.double(), x.double())
    wt = w.t().contiguous()
    for y in (ops.gemm(lib, x, w)[0], ops.gemm(lib, x, wt, transposed=True)[0]):
        assert _rel(y, z) < 2e-7
        assert float((y - z).mean().abs() / z.norm() * z.numel() ** 0.5) < 3e-9
    y, zk = ops.gemm(lib, x, w, bias, res, "gelu", keep_z=True)
    assert _rel(zk, z) < 2e-7 and _rel(y, F.gelu(z + bias.double()[:, None]) + res.double()) < 5e-7
    gw, gb = ops.weight_grad(lib, g, x, need_bias_grad=True)
    assert _rel(gw, torch.matmul(g.double(), x.double().transpose(1, 2)).sum(0)) < 6e-7
    assert _rel(gb, g.double().sum((0, 2))) < 4e-6


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-36, 1e-20, 1e30])
def test_parts_of_small_and_large_values(scale):
    lib, (x, _, _, g), w, _ = _setup("cuda", (2, 72, 30, 20003), torch.float32)
    x *= scale
    assert _rel(ops.gemm(lib, x, w)[0], torch.matmul(w.double(), x.double())) < 4e-7
    gw, _ = ops.weight_grad(lib, g, x)
    assert _rel(gw, torch.matmul(g.double(), x.double().transpose(1, 2)).sum(0)) < 1e-6


def _each_within(y, a, b):
    """Every sum within what a chain of float32 sums may be off (and the least normal number), that of nothing but zeros
    zero."""
    want, size = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    off = (y.double() - want).abs() - size * (b.size(-2) + 8) * 2.0 ** -24
    assert bool((off <= 2.0 ** -126).all()) and bool((y[size == 0] == 0).all())


# exponents of x's even and odd voxels, of w's rows 1 and 2, and of w (or g in its place)
@pytest.mark.gpu
@pytest.mark.parametrize("voxels,rows,weight", [((0, -118), 0, 0), ((-118, -118), 0, 40), ((-140, -140), 0, 70), ((0, 0), -115, 0),
                                                ((0, -60), -45, 0), ((90, 90), -118, 0), ((0, -500), -500, 0)])
def test_parts_of_values_of_very_different_sizes(voxels, rows, weight):
    """Small values beside others, and against large ones: bf16 parts of them are denormal, or their products' are."""
    print("case", voxels, rows, weight, flush=True)
    lib, (x, _, _, g), w, _ = _setup("cuda", (2, 72, 130, 20003), torch.float32)
    x[..., 0::2] *= 2.0 ** voxels[0]
    x[..., 1::2] *= 2.0 ** voxels[1]
    for t in (w, g.transpose(0, 1)):
        t *= 2.0 ** weight
        t[1:3] *= 2.0 ** rows
    x[:, 4] = 0
    for y in (ops.gemm(lib, x, w)[0], ops.gemm(lib, x, w.t().contiguous(), transposed=True)[0]):
        _each_within(y, w, x)
    gw, _ = ops.weight_grad(lib, g, x)
    _each_within(gw, g.transpose(0, 1).flatten(1), x.transpose(0, 1).flatten(1).t())


@pytest.mark.gpu
@pytest.mark.parametrize("one,size,weight", [(3.4e38, 0, -100), (3.4e38, -120, -20), (1.0, 64, 56), (1.0, 50, 64)])
def test_parts_of_values_near_the_largest(one, size, weight):
    """A value that rounds to an infinite bf16, beside others and small weights, and products of which a few sums would pass
    the largest float32 on the way."""
    print("case", one, size, weight, flush=True)
    lib, (x, _, _, g), w, _ = _setup("cuda", (2, 72, 130, 20003), torch.float32)
    x *= 2.0 ** size
    x[0, 3, 7] = one
    w *= 2.0 ** weight
    g *= 2.0 ** (weight - 8)
    for y in (ops.gemm(lib, x, w)[0], ops.gemm(lib, x, w.t().contiguous(), transposed=True)[0]):
        _each_within(y, w, x)
    gw, _ = ops.weight_grad(lib, g, x)
    _each_within(gw, g.transpose(0, 1).flatten(1), x.transpose(0, 1).flatten(1).t())


@pytest.mark.gpu
def test_parts_of_values_that_are_not_finite():
    """What a float32 product makes of infinities, NaN and values beyond the range of bf16: an infinity's column is
    infinite by the weight's sign, the rest finite."""
    lib, (x, _, _, g), w, _ = _setup("cuda", (2, 72, 30, 20003), torch.float32)
    x[0, 3, 7], x[0, 71, 20002], x[1, 5, 130], x[1, 6, 131] = float("inf"), float("-inf"), float("nan"), 3.4e38
    for y, want in ((ops.gemm(lib, x, w)[0], torch.matmul(w.double(), x.double())),
                    (ops.weight_grad(lib, g, x)[0], torch.matmul(g.double(), x.double().transpose(1, 2)).sum(0))):
        want = want.float()
        assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isinf(), want.isinf())
        assert torch.equal(y[y.isinf()], want[want.isinf()])
        ok = want.isfinite() & (want.abs() < 1e30)
        assert _rel(y[ok], want[ok]) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("transposed", [False, True])
def test_more_samples_than_a_launch_has_threads_for(transposed):
    """2^20 samples of a voxel into 1040 channels: 2^32 threads and more, those of the last launch's samples included."""
    print("case", transposed, flush=True)
    lib, B, cout = _lib.get_library(), 1 << 20, 1040
    gen = torch.Generator(device="cuda").manual_seed(0)
    x, w, bias = (torch.randn(*s, generator=gen, device="cuda") for s in ((B, 1, 1), (cout, 1), (cout,)))
    y, _ = ops.gemm(lib, x, w.t().contiguous() if transposed else w, bias, None, transposed=transposed)
    want = torch.addcmul(bias[:, None], w, x)
    assert float((y - want).abs().max()) < 2e-5        # (products of up to 30)
    assert bool((y[-16:] != 0).any(dim=(1, 2)).all())


def test_refused_arguments():
    lib = hostcheck_library()
    x, w = torch.zeros(1, 8, 4), torch.zeros(6, 8)
    with pytest.raises(_lib.NdcError):      # an activation reads W as rows
        ops.gemm(lib, x, w.t().contiguous(), act="relu", transposed=True)
    with pytest.raises(_lib.NdcError):      # the gradient mode reads its transpose
        ops.gemm(lib, x, w, residual=torch.zeros(1, 6, 4), act="gelu_grad")
    with pytest.raises(_lib.NdcError):      # and needs the pre-activation
        ops.gemm(lib, x, w.t().contiguous(), act="gelu_grad", transposed=True)
