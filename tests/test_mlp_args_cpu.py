"""What the entry points of the MLP on chip ask of their addresses, on the host build (which has no
sequential form of these kernels: a call that gets past the checks ends in its own status)."""

import ctypes

import pytest

from deconver_amd import _lib
from tests.helpers import hostcheck_library

WORKSPACE, NO_KERNEL = -4, -2


def _call(name, w1, w2, w_dtype):
    dll = hostcheck_library()._dll
    c, n = 32, 64
    buf = ctypes.create_string_buffer(1 << 20)
    base = (ctypes.addressof(buf) + 255) // 256 * 256
    vp, i64 = ctypes.c_void_p, ctypes.c_int64
    at = [vp(base + 65536 * i) for i in range(8)]
    w1, w2 = vp(at[6].value + w1), vp(at[7].value + w2)
    if name == "forward":
        return dll.ndc_mlp_forward(at[0], None, w1, w2, w_dtype, None, None, None, at[1], i64(1), i64(c), i64(n), _lib.NDC_BF16, None)
    dll.ndc_mlp_workspace_bytes.restype = ctypes.c_size_t
    need = dll.ndc_mlp_workspace_bytes(i64(1), i64(c), i64(n))
    return dll.ndc_mlp_backward(at[0], at[1], w1, w2, w_dtype, None, at[2], at[3], None, at[4], None, i64(1), i64(c), i64(n),
                                _lib.NDC_BF16, at[5], ctypes.c_size_t(need), None)


@pytest.mark.parametrize("name", ["forward", "backward"])
@pytest.mark.parametrize("w1,w2,w_dtype,status", [
    (0, 0, _lib.NDC_F32, NO_KERNEL), (4, 4, _lib.NDC_F32, NO_KERNEL), (2, 0, _lib.NDC_F32, WORKSPACE), (0, 2, _lib.NDC_F32, WORKSPACE),
    (2, 2, _lib.NDC_BF16, NO_KERNEL), (1, 0, _lib.NDC_BF16, WORKSPACE), (0, 3, _lib.NDC_BF16, WORKSPACE)])
def test_weights_are_aligned_to_an_element(name, w1, w2, w_dtype, status):
    assert _call(name, w1, w2, w_dtype) == status
