"""A frame that is refused by its parameters still leaves the caller's arrays
cleared (RGB 127, ids -1, as the reference clears its output before a frame,
RayTracer.cpp:620), never the pixels of a frame rendered before it."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import log

pytestmark = pytest.mark.gpu

W, H = 64, 48


@pytest.mark.parametrize("what,kw", [("unknown mode", dict(mode=0x40)), ("re-test in the megakernel", dict(engine=1, flags=1)),
                                     ("re-test of a primary-only mode", dict(mode=0x2, flags=1))], ids=lambda v: v if isinstance(v, str) else "")
def test_refused_frame_leaves_cleared_outputs(rt_gpu, what, kw):
    rt = rt_gpu
    lib = rt._capi.load()
    log(f"case: {what}")
    ds = rt.DeviceScene(rt.HostScene.workload(1))
    ds.render(rt.params(W, H, max_level=2))  # what must not come back
    p = rt.params(W, H, max_level=2, **kw)
    rgb, ids = np.zeros((H, W, 3), np.uint8), np.zeros((H, W, 2), np.int32)
    at = lambda a: a.ctypes.data_as(C.c_void_p)
    assert lib.rtg_render(ds.h, C.byref(p), at(rgb), at(ids), None, None) == -1
    assert (rgb == 127).all() and (ids == -1).all()
    hip = C.CDLL("libamdhip64.so.7")  # the runtime librtg loaded
    out, got = C.c_void_p(), np.zeros((H, W, 3), np.uint8)
    assert hip.hipMalloc(C.byref(out), C.c_size_t(got.nbytes)) == 0
    assert hip.hipMemcpy(out, at(got), C.c_size_t(got.nbytes), 1) == 0
    assert lib.rtg_render_device(ds.h, C.byref(p), out, None, None, None, None) == -1
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemcpy(at(got), out, C.c_size_t(got.nbytes), 2) == 0
    assert hip.hipFree(out) == 0
    assert (got == 127).all()
