"""Channel-first helper layers around the NDC update (``deconver/layers`` of the reference):
``Linear`` (1x1 projection, parameters held by an ``nn.Conv1d`` as there), ``MLP``,
``LayerNorm``, and the network's resampling convolutions, head and stem as subclasses of the
``torch.nn`` convolutions.  On the GPU the projections are channel-first GEMMs
with bias, activation and residual sum in their epilogues (the HIP library's streaming and tiled
ones; the library GEMM through ``torch.bmm`` where it is ahead);
the strided convolutions are a regrouping copy in front of the same
projection.  Parameter names and shapes match the reference, so its checkpoints load
unchanged."""

from __future__ import annotations

import math
from typing import Optional

import torch
from torch import nn
from torch.nn.modules.utils import _pair

from . import _lib, ops


_ACT_TAGS = {None: _lib.ACT_NONE, "relu": _lib.ACT_RELU, "gelu": _lib.ACT_GELU}
_ACT_FUNCTIONS = {None: lambda t: t, "relu": torch.relu, "gelu": torch.nn.functional.gelu}


def pointwise_linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
                     act: Optional[str] = None, residual: Optional[torch.Tensor] = None,
                     grad_premasked: bool = False, transposed: bool = False) -> torch.Tensor:
    """``act(W x + bias) + residual``: the 1x1 projection ``(B, Cin, N) -> (B, Cout, N)`` with
    ``weight`` of shape ``(Cout, Cin)`` or ``(Cout, *)`` with ``Cin`` elements per row (with
    ``transposed``: the ``(Cin, Cout)`` storage of it), optionally followed by an activation (``"relu"`` or ``"gelu"``, the exact one) and the sum with a tensor of the
    output's shape.  bfloat16 (stored or under autocast) and float32 tensors on the GPU run as
    GEMMs on the channel-first layout, with the tail in the epilogue of the HIP library's own GEMMs or
    as one pass of it over a library GEMM's result (``choose_gemm`` in ``csrc/ndc_torch.cpp`` says
    which); everything else as the reference's ``conv1d`` followed by PyTorch's activation and sum.

    ``grad_premasked`` (GEMM route, ``act="relu"`` without residual only; ignored elsewhere): the
    caller guarantees that every gradient reaching the result is already zero where the result
    is -- its only consumer took it through the rectifier (``Deconv.forward(rectified_input=True)``)
    --, so the backward skips the rectifier's pass."""
    dtype = x.dtype
    if x.is_cuda and torch.is_autocast_enabled(x.device.type):
        dtype = torch.get_autocast_dtype(x.device.type)
    # (2-D network in float32, batch 8: 16.6 ms per step this way against 20.8 ms with the
    # GEMM left to the library's conv1d, whose weight gradient goes through layout transposes)
    if not x.is_cuda or x.dim() != 3 or dtype not in (torch.bfloat16, torch.float32):
        w = weight.t() if transposed else weight.flatten(1)
        y = _ACT_FUNCTIONS[act](torch.nn.functional.conv1d(x, w.unsqueeze(-1), bias))
        return y if residual is None else residual + y
    return _lib.get_native().linear(x if x.dtype == dtype else x.to(dtype), weight, bias, _ACT_TAGS[act], residual,
                                    grad_premasked, transposed)


def _gemm_route(x: torch.Tensor) -> bool:
    """True for the tensors whose 1x1 projection ``pointwise_linear`` runs as channel-first
    GEMMs: bfloat16 (stored or under autocast) and float32 on the GPU."""
    dtype = x.dtype
    if x.is_cuda and torch.is_autocast_enabled(x.device.type):
        dtype = torch.get_autocast_dtype(x.device.type)
    return x.is_cuda and dtype in (torch.bfloat16, torch.float32)


def _is_patch_conv(conv) -> bool:
    """A convolution whose windows tile the input: stride == kernel size, no padding, no
    dilation, one group (and no output padding on a transposed one)."""
    return (tuple(conv.stride) == tuple(conv.kernel_size) and all(p == 0 for p in conv.padding)
            and all(d == 1 for d in conv.dilation) and conv.groups == 1
            and isinstance(conv.padding, tuple)
            and all(p == 0 for p in getattr(conv, "output_padding", ())))


def patches_to_channels(x: torch.Tensor, k) -> torch.Tensor:
    """``(B, C, *S) -> (B, C * prod(k), prod(S // k))``: every ``k`` window of the grid becomes
    one column, channel-major then window offset (the order of a convolution weight's
    ``(Cin, *k)`` axes).  Rows and planes that do not fill a window are dropped, as a strided
    convolution drops them."""
    B, C = x.shape[:2]
    nd = len(k)
    if all(v == 1 for v in k):
        return x.flatten(2)
    coarse = [s // v for s, v in zip(x.shape[2:], k)]
    if any(c * v != s for c, v, s in zip(coarse, k, x.shape[2:])):
        x = x[(slice(None), slice(None), *[slice(0, c * v) for c, v in zip(coarse, k)])]
    split = [B, C]
    for c, v in zip(coarse, k):
        split += [c, v]
    x = x.reshape(split)
    order = [0, 1] + [3 + 2 * i for i in range(nd)] + [2 + 2 * i for i in range(nd)]
    return x.permute(order).reshape(B, C * math.prod(k), math.prod(coarse))


def channels_to_patches(y: torch.Tensor, k, coarse) -> torch.Tensor:
    """Inverse of ``patches_to_channels`` on an exactly tiled grid:
    ``(B, C * prod(k), prod(coarse)) -> (B, C, *(coarse * k))``."""
    B = y.shape[0]
    nd = len(k)
    C = y.shape[1] // math.prod(k)
    if all(v == 1 for v in k):
        return y.view(B, C, *coarse)
    y = y.view(B, C, *k, *coarse)
    order = [0, 1]
    for i in range(nd):
        order += [2 + nd + i, 2 + i]
    return y.permute(order).reshape(B, C, *[c * v for c, v in zip(coarse, k)])


def _regroup_on_hip(fine_shape, dtype, k, *tensors) -> bool:
    """2-windows in every dimension and GPU buffers the kernel takes (``tensors``: the ones
    that exist already)."""
    return (all(v == 2 for v in k) and len(k) in (2, 3) and all(t.is_cuda for t in tensors)
            and ops.regroup2_applies(tuple(fine_shape), dtype, *[t.data_ptr() for t in tensors]))


def patch_conv(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
    """``conv(x, weight, bias, stride=weight.shape[2:])``, no padding: a strided convolution
    whose windows tile its input is a regrouping of the grid followed by the 1x1 projection."""
    k = tuple(weight.shape[2:])
    coarse = [s // v for s, v in zip(x.shape[2:], k)]
    if x.is_cuda and torch.is_autocast_enabled(x.device.type):
        x = x.to(torch.get_autocast_dtype(x.device.type))     # before the regrouping, not after
    xc = x.contiguous()
    if _regroup_on_hip(xc.shape, xc.dtype, k, xc):
        cols = _lib.get_native().regroup(xc, True, None).flatten(2)
    else:
        cols = patches_to_channels(x, k)
    y = pointwise_linear(cols, weight, bias)
    return y.view(x.shape[0], -1, *coarse)


def patch_conv_transpose(x: torch.Tensor, weight: torch.Tensor,
                         bias: Optional[torch.Tensor]) -> torch.Tensor:
    """``conv_transpose(x, weight, bias, stride=weight.shape[2:])``: the 1x1 projection to
    ``Cout * prod(k)`` channels, then every column spread over its window of the finer grid."""
    k = tuple(weight.shape[2:])
    # weight (Cin, Cout, *k): row (cout, offset) of the projection is weight[:, cout, offset]
    w = weight.flatten(1)
    fine = (x.shape[0], weight.shape[1], *[s * v for s, v in zip(x.shape[2:], k)])
    dtype = x.dtype
    if x.is_cuda and torch.is_autocast_enabled(x.device.type):
        dtype = torch.get_autocast_dtype(x.device.type)
    if x.is_cuda and _regroup_on_hip(fine, dtype, k):
        # the bias rides on the regrouping pass
        y = pointwise_linear(x.flatten(2), w, None, transposed=True).contiguous()
        if _regroup_on_hip(fine, y.dtype, k, y):
            return _lib.get_native().regroup(y.view(x.shape[0], -1, *x.shape[2:]), False, bias)
        y = channels_to_patches(y, k, x.shape[2:])
        return y if bias is None else y + bias.to(y.dtype).view(1, -1, *([1] * len(k)))
    if bias is not None:
        bias = bias.repeat_interleave(math.prod(k))
    return channels_to_patches(pointwise_linear(x.flatten(2), w, bias, transposed=True), k, x.shape[2:])


class _PatchConvMixin:
    """The network's 2-tap resampling convolutions (unet.py:36-60) and its 1-tap head are
    convolutions whose windows tile the input.  bfloat16 and float32 tensors on the GPU take
    the form of ``patch_conv`` here -- one regrouping copy and the projection of
    ``pointwise_linear`` instead of the library's column-matrix convolution; everything else,
    and any other stride or padding, runs the parent class's convolution.  Parameters, their
    shapes and names are the parent's."""

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if _is_patch_conv(self) and _gemm_route(x) and x.dim() == len(self.kernel_size) + 2:
            return patch_conv(x, self.weight, self.bias)
        return super().forward(x)


class _PatchConvTransposeMixin:
    """The transposed counterpart (unet.py:108-131), as ``patch_conv_transpose``."""

    def forward(self, x: torch.Tensor, output_size=None) -> torch.Tensor:
        if (output_size is None and _is_patch_conv(self) and _gemm_route(x)
                and x.dim() == len(self.kernel_size) + 2):
            return patch_conv_transpose(x, self.weight, self.bias)
        return super().forward(x, output_size)


def unfold_conv(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
    """``conv(x, weight, bias, stride=1, padding=k // 2)`` for odd kernel sizes ``k`` as a column
    matrix (every tap's shifted copy of the zero-padded input, channel-major then tap: the order
    of the weight's ``(Cin, *k)`` axes) followed by the 1x1 projection.  An input that needs no
    gradient -- images -- has the matrix made by one launch."""
    k = tuple(weight.shape[2:])
    size = x.shape[2:]
    if (x.is_cuda and len(k) <= 3 and x.dtype in (torch.bfloat16, torch.float32) and x.numel() > 0
            and math.prod(size) < 2 ** 31 and not (torch.is_grad_enabled() and x.requires_grad)
            and not torch.jit.is_tracing()):     # (what is traced runs on other inputs)
        cols = _lib.get_native().columns(x.contiguous(), list(k))
        return pointwise_linear(cols, weight, bias).view(x.shape[0], -1, *size)
    pad = []
    for v in reversed(k):
        pad += [v // 2, v // 2]
    xp = torch.nn.functional.pad(x, pad)
    shifts = [()]
    for v in k:
        shifts = [t + (o,) for t in shifts for o in range(v)]
    cols = torch.stack([xp[(slice(None), slice(None), *[slice(o, o + n) for o, n in zip(t, size)])]
                        for t in shifts], dim=2)
    y = pointwise_linear(cols.flatten(1, 2).flatten(2), weight, bias)
    return y.view(x.shape[0], -1, *size)


class _UnfoldConvMixin:
    """The network's stem (unet.py:175-276: a 3-tap convolution from the few image channels to
    the first width): with few input channels the column matrix is small next to the output,
    and bfloat16 / float32 tensors on the GPU take ``unfold_conv`` -- one gather and the
    projection of ``pointwise_linear`` -- instead of the library's convolution, whose weight
    gradient alone takes longer.  Anything else (more than ``max_columns`` rows in the column matrix, other
    strides or paddings) runs the parent class's convolution."""

    max_columns = 128

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        k = tuple(self.kernel_size)
        if (_gemm_route(x) and x.dim() == len(k) + 2 and all(v % 2 == 1 for v in k)
                and isinstance(self.padding, tuple) and tuple(self.padding) == tuple(v // 2 for v in k)
                and all(v == 1 for v in self.stride) and all(v == 1 for v in self.dilation)
                and self.groups == 1 and self.padding_mode == "zeros"
                and self.in_channels * math.prod(k) <= self.max_columns):
            if torch.is_autocast_enabled(x.device.type):
                x = x.to(torch.get_autocast_dtype(x.device.type))    # before the gather, not after
            return unfold_conv(x, self.weight, self.bias)
        return super().forward(x)


class UnfoldConv1d(_UnfoldConvMixin, nn.Conv1d):
    pass


class UnfoldConv2d(_UnfoldConvMixin, nn.Conv2d):
    pass


class UnfoldConv3d(_UnfoldConvMixin, nn.Conv3d):
    pass


class PatchConv1d(_PatchConvMixin, nn.Conv1d):
    pass


class PatchConv2d(_PatchConvMixin, nn.Conv2d):
    pass


class PatchConv3d(_PatchConvMixin, nn.Conv3d):
    pass


class PatchConvTranspose1d(_PatchConvTransposeMixin, nn.ConvTranspose1d):
    pass


class PatchConvTranspose2d(_PatchConvTransposeMixin, nn.ConvTranspose2d):
    pass


class PatchConvTranspose3d(_PatchConvTransposeMixin, nn.ConvTranspose3d):
    pass


_any_global_hook = nn.modules.module._has_any_global_hook


def _hooked(*modules: nn.Module) -> bool:
    """Whether a hook watches a call of one of ``modules`` (or of every module): a caller that runs a
    module's work inside another call then calls the module instead."""
    if _any_global_hook():
        return True
    for m in modules:       # (a loop: twice as fast as any() over a generator, five times in a block's call)
        if m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks:
            return True
    return False


class Linear(nn.Module):
    """Pointwise linear map over channels for ``(N, C, *)`` inputs (layers/linear.py:34-58).

    The weight lives in ``self.linear`` (an ``nn.Conv1d`` with kernel size 1), hence the
    state-dict keys ``linear.weight`` ``(Cout, Cin, 1)`` and ``linear.bias``.
    """

    def __init__(self, in_channels: int, out_channels: int, bias: bool = True,
                 device: Optional[torch.device] = None, dtype: Optional[torch.dtype] = None):
        super().__init__()
        self.flatten = nn.Flatten(start_dim=2)
        self.linear = nn.Conv1d(in_channels, out_channels, kernel_size=1, bias=bias,
                                device=device, dtype=dtype)

    def forward(self, x: torch.Tensor, act: Optional[str] = None,
                residual: Optional[torch.Tensor] = None, grad_premasked: bool = False) -> torch.Tensor:
        """``act(linear(x)) + residual``; ``act`` None, ``"relu"`` or ``"gelu"``; ``residual``
        of the output's shape; ``grad_premasked`` as for ``pointwise_linear``."""
        shape = x.shape
        if residual is not None:
            residual = residual.flatten(2)
        y = pointwise_linear(self.flatten(x), self.linear.weight, self.linear.bias, act, residual,
                             grad_premasked)
        return y.view(shape[0], -1, *shape[2:])


class MLP(nn.Module):
    """Linear - GELU - Linear on channels, with dropout after each (layers/mlp.py:40-63)."""

    def __init__(self, in_channels: int, out_channels: Optional[int] = None,
                 hidden_channels: Optional[int] = None, ratio: float = 4.0,
                 dropout: float | tuple[float, float] = 0.0, **kwargs):
        super().__init__()
        out_channels = out_channels or in_channels
        hidden_channels = hidden_channels or int(ratio * in_channels)
        p_hidden, p_out = _pair(dropout)
        self.block = nn.Sequential(
            Linear(in_channels, hidden_channels, **kwargs),
            nn.GELU(),
            nn.Dropout(p_hidden),
            Linear(hidden_channels, out_channels, **kwargs),
            nn.Dropout(p_out),
        )

    def forward(self, x: torch.Tensor, residual: Optional[torch.Tensor] = None) -> torch.Tensor:
        """``block(x)``, plus ``residual`` if given.  With the exact GELU and no active dropout
        the activation and the sum ride on the projections (``Linear.forward``); parts that are hooked
        or of another class are called one by one."""
        block = self.block
        first, act, drop1, second, drop2 = block
        idle = lambda d: d.p == 0 or not d.training   # noqa: E731
        if (type(first) is Linear and type(second) is Linear and type(act) is nn.GELU
                and act.approximate == "none" and idle(drop1) and idle(drop2)
                and not _hooked(block, first, act, drop1, second, drop2)):
            fused = self._fused(first, second, x, residual)
            return second(first(x, act="gelu"), residual=residual) if fused is None else fused
        y = block(x)
        return y if residual is None else residual + y

    @staticmethod
    def _fused(first: "Linear", second: "Linear", x: torch.Tensor, residual: Optional[torch.Tensor]):
        """The block as one compiled node (the hidden tensor's gradient is written once and, where the
        library's own GEMMs make it, never read back by an activation pass) for bfloat16 (stored or
        under autocast) and float32 tensors on the GPU, else None."""
        if not _gemm_route(x):
            return None
        dtype = torch.get_autocast_dtype(x.device.type) if torch.is_autocast_enabled(x.device.type) else x.dtype
        w1, w2 = first.linear.weight, second.linear.weight
        flat = x.flatten(2)
        if flat.dtype != dtype:
            flat = flat.to(dtype)
        y = _lib.get_native().mlp(flat, w1, first.linear.bias, w2, second.linear.bias,
                                  None if residual is None else residual.flatten(2))
        return y.view(x.shape[0], w2.shape[0], *x.shape[2:])


_CHNORM_MIN_VOXELS = 32768


class LayerNorm(nn.Module):
    """``nn.LayerNorm`` over the channel axis of a ``(B, C, *S)`` tensor (layers/norm.py:25-34).

    The reference moves the channel axis last, normalises and moves it back, which costs two
    generic strided copies (the norm's own and the next projection's ``contiguous()``).  On the
    GPU (float32 / bfloat16 tensors) the HIP kernels normalise over the channel axis where it
    is; parameters and state dict are ``nn.LayerNorm``'s, and under autocast the arithmetic and
    the result are float32, as PyTorch's autocast rules make them for the reference."""

    def __init__(self, dim: int, **kwargs):
        super().__init__()
        self.norm = nn.LayerNorm(dim, **kwargs)

    def _hip(self, x: torch.Tensor) -> Optional[torch.Tensor]:
        """The normalised ``x`` from the HIP kernels, in its own type, or None if they do not take it."""
        if not (x.is_cuda and x.dim() >= 3 and len(self.norm.normalized_shape) == 1 and x.numel() > 0
                and x.shape[1] == self.norm.normalized_shape[0] and x.dtype in (torch.float32, torch.bfloat16)):
            return None
        y = _lib.get_native().channel_norm(x.flatten(2), self.norm.weight, self.norm.bias, float(self.norm.eps))
        return y.view(x.shape)

    def _widened(self, x: torch.Tensor) -> torch.Tensor:
        return x.float() if x.is_cuda and torch.is_autocast_enabled(x.device.type) else x

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        # (below 32 768 voxels in all a caller gets the reference's form, a view of a channels-last result)
        y = None
        if x.is_cuda and x.dim() >= 3 and x.shape[0] * x[0, 0].numel() >= _CHNORM_MIN_VOXELS:
            y = self._hip(self._widened(x))
        return self.norm(x.movedim(1, -1)).movedim(-1, 1) if y is None else y

    def for_projection(self, x: torch.Tensor, *consumers: nn.Module) -> torch.Tensor:
        """``forward(x)`` for a caller that hands it to a projection (``consumers``: it, and the module
        around it that is called), which wants it channel-first and, under bfloat16 autocast, rounded to
        bfloat16: the kernels at every size, and bfloat16 values under bfloat16 autocast normalised (in
        float32 arithmetic) and rounded in one pass -- the bits that widening, normalising and rounding
        in three passes over twice the bytes give, in both directions.  Hooks see what ``forward`` makes."""
        y = None
        if (type(self) is LayerNorm and type(self.norm) is nn.LayerNorm and _gemm_route(x)
                and not _hooked(self, self.norm, *consumers)):
            narrow = (x.dtype == torch.bfloat16 and torch.is_autocast_enabled(x.device.type)
                      and torch.get_autocast_dtype(x.device.type) == torch.bfloat16)
            y = self._hip(x if narrow else self._widened(x))
        return self(x) if y is None else y
