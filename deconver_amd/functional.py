"""Autograd node of one NDC source update, running on the HIP kernels.

Mirrors ``deconver/deconvolution/functional.py:97-207`` of the reference
(``DeconvUpdate`` / ``deconv_update``): same arguments, same returned gradients
``(gx, gz, gh, gb, None x5)``, same refusal of double backward.  It saves the reference's
``(x, z, t1, h, bias)`` plus, unless ``save_ratio(False)`` was called, the forward's
``s/(A(t1)+eps)`` and ``(A(x)+eps)/(A(t1)+eps)``: two tensors of the size of the output
kept until backward, which then does not gather ``A(x)`` and ``A(t1)`` a second time.
The arithmetic is in ``libdeconver_ndc.so``, the node in ``_native.so``; there is no PyTorch
implementation behind it.
"""

from __future__ import annotations

import os
from typing import Optional

import torch
from torch import Tensor

from . import _lib, ops

__all__ = ["deconv_update", "projected_update", "hip_kernels_apply", "DeconvUpdate", "save_ratio", "matrix_kernels"]

_SAVE_RATIO = os.environ.get("DECONVER_NDC_SAVE_RATIO", "1") != "0"


def save_ratio(enabled: Optional[bool] = None) -> bool:
    """Get or set whether training keeps the forward's denominator and ratio for backward.

    On (the default; environment ``DECONVER_NDC_SAVE_RATIO=0`` turns it off): each update
    node holds two more tensors of the size of its output until backward, and backward is
    shorter.  Off: backward re-gathers them from ``x`` and ``t1`` as the reference does.
    """
    global _SAVE_RATIO
    if enabled is not None:
        _SAVE_RATIO = bool(enabled)
    return _SAVE_RATIO


def matrix_kernels(enabled: Optional[bool] = None) -> bool:
    """Get or set whether bf16 3x3x3 updates may run on the kernels that use the 4x4x4 matrix
    instruction (the process default, ``ndc_matrix_kernels``).  Off by default (environment
    ``DECONVER_NDC_MATRIX=1`` turns it on when the library is loaded): the path is specified
    without matrix instructions.  Same results to the bf16 tolerance, less time per step.
    An update node reads the setting once, in its forward, and names the family in its forward
    and backward calls (``ndc_geom.path``), so a change takes effect from the next forward."""
    return _lib.get_library().matrix_kernels(enabled)


def hip_kernels_apply(x: Tensor, m: int, sc: int, kernel_size, dtype=None) -> bool:
    """Whether the HIP update can run for this input and filter geometry.

    Counterpart of ``fused_kernels_apply`` (``functional.py:34-47``): device tensors only,
    no active functorch transform, float32 or bfloat16 storage, rank 1-3, odd kernel.
    """
    try:
        functorch = torch._C._are_functorch_transforms_active()
    except AttributeError:  # pragma: no cover
        functorch = False
    dtype = x.dtype if dtype is None else dtype
    if functorch or not x.is_cuda or dtype not in (torch.float32, torch.bfloat16):
        return False
    if not 1 <= len(kernel_size) <= 3 or x.dim() - 2 != len(kernel_size):
        return False
    if any(k % 2 == 0 for k in kernel_size):
        return False
    lib = _lib.get_library()  # raises when the library is missing: no silent fallback
    g = _lib.make_geom(x.shape[0], x.shape[1] // m, m, sc, x.shape[2:], kernel_size,
                       ops.dtype_tag(dtype), True, 0.0)
    return lib.check_geometry(g) == 0


class DeconvUpdate:
    """``out = relu(z + b) * (A(x) + eps) / (A(K(relu(z + b))) + eps)`` as an autograd node, called
    through ``apply`` as the reference's ``Function`` is (functional.py:97-182).

    The node itself is compiled (``csrc/ndc_torch.cpp``).  Channels-last tensors
    (torch.channels_last / channels_last_3d) come in through the library's tiled transposition,
    and results and gradients go back out the same way, in the layout of the tensor they belong
    to.  A second differentiation is refused."""

    @staticmethod
    def apply(x, z, h, bias, groups, m, sc, eps, relu_input, taps=None):
        if not x.is_cuda:
            raise RuntimeError("deconv_update runs on the GPU only (HIP kernels); "
                               "CPU tensors take the layer's general PyTorch path")
        return _lib.get_native().update(x, z, h, bias, groups, m, sc, eps, relu_input, taps, _SAVE_RATIO)


def deconv_update(x: Tensor, z: Tensor, h: Tensor, bias: Optional[Tensor], *, groups: int,
                  m: int, sc: int, eps: float, relu_input: bool,
                  taps: Optional[Tensor] = None) -> Tensor:
    """One multiplicative source update.

    Args:
        x: input, ``(B, C, *S)``.
        z: projection output ``(B, groups*sc, *S)``, pre-bias and pre-ReLU on the first
            iteration (the kernels apply both on load); the rectified source afterwards.
        h: rectified filter ``(C, sc, *k)``, float32.
        bias: the projection's bias (float32) or ``None``.
        eps: stabiliser added to numerator and denominator.
        taps: optional (not in the reference): the table ``ops.prepare_taps`` made for this
            ``h``, for callers that run several updates with one filter; made here otherwise.
    """
    return DeconvUpdate.apply(x, z, h, bias, groups, m, sc, eps, relu_input, taps)


def projected_update(x: Tensor, weight: Tensor, h: Tensor, bias: Optional[Tensor], *, groups: int,
                     m: int, sc: int, eps: float, taps: Optional[Tensor] = None,
                     rectified_input: bool = False, rectify_filter: bool = False) -> Tensor:
    """``deconv_update(x, W x, h, bias, relu_input=True)`` as one autograd node (not in the
    reference, which records the projection and the update separately).

    One node instead of two because ``x`` feeds both the projection and the update: as two
    nodes their input gradients are two tensors that autograd adds in a pass of its own;
    here the projection's input-gradient GEMM accumulates onto the update's ``gx``
    (``gx += W^T gz``, one rounding instead of two in bfloat16).

    Args:
        x: input ``(B, C, *S)``, float32 or bfloat16 on the GPU, in any layout (channels-last tensors
            come in through the library's tiled transposition, and their gradient goes back so).
        weight: the projection's weight ``(groups*sc, C)``, any floating dtype (cast to ``x``'s
            for the GEMMs; its gradient comes back in its own dtype).
        h, bias, groups, m, sc, eps, taps: as for ``deconv_update``.
        rectified_input: ``x`` is the output of a rectifier whose backward pass its producer
            skips (``Linear(..., act="relu", grad_premasked=True)``): the gradient of ``x`` is
            returned zero where ``x`` is, from the GEMM that forms it.
        rectify_filter: ``h`` is the filter before its rectifier; the node applies it, and returns
            the gradient of the unrectified filter.
    """
    return _lib.get_native().projected_update(x, weight, h, bias, groups, m, sc, eps, taps, rectified_input,
                                              rectify_filter, _SAVE_RATIO)
