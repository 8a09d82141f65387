"""What a thread keeps of its launch plans: sizes that share a slot, more sizes than are kept, threads."""

import ctypes
import threading

import torch

from deconver_amd import ops
from tests.helpers import hostcheck_library


def _answers(lib, shapes):
    out = []
    for dtype, channels, size in shapes:
        x = torch.empty(1, channels, *size, dtype=dtype, device="meta")
        h = torch.empty(channels, 4, *((3,) * 3 if len(size) == 3 else (5, 5)))
        g = ops.make_geom_for(x, h, channels, 1, 4, 1e-8, True)
        r = ctypes.byref(g)
        d = lib._dll
        out.append((d.ndc_fused_supported(r), d.ndc_backward_uses_saved(r), d.ndc_taps_bytes(r), d.ndc_forward_workspace_bytes(r),
                    d.ndc_backward_workspace_bytes(r, 1, 1, 1, 1)))
    return out


def test_kept_plans_are_of_the_sizes_asked_for():
    lib = hostcheck_library()
    shapes = [(t, c, s) for t in (torch.float32, torch.bfloat16) for c in (1, 32)
              for s in [(8 + i, 12, 16 + i % 5) for i in range(40)] + [(9 + i, 20) for i in range(40)]]
    results = {}

    def first_of_each(i):      # (a thread has kept nothing yet)
        results[i] = _answers(lib, [shapes[i]])[0]

    for i in range(len(shapes)):
        t = threading.Thread(target=first_of_each, args=(i,))
        t.start()
        t.join()
    want = [results[i] for i in range(len(shapes))]
    assert len(set(want)) > 20
    for order in (shapes, shapes[::-1], shapes[::2] + shapes[1::2]):
        back = dict(zip(map(str, order), _answers(lib, order)))
        assert [back[str(s)] for s in shapes] == want
