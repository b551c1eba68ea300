"""Device memory the library's queues take for a frame: what its kernels read
and no more.  In a process of its own, whose workspace is empty at the start."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

from conftest import ROOT, log

pytestmark = pytest.mark.gpu

W, H = 1920, 1080
SAMPLES = W * H  # whole 8x8 blocks
HIT, RAY, NODE, MASK, SHADOW, COLOUR = 48, 48, 64, 4, 4, 16  # bytes; HIT with the child's source copy

# a 1080p frame after a 64x64 one of the same kind, which takes all that does not grow with the frame
PROGRAM = """
import ctypes as C, sys
import raytrace_amd as rt
rt.init(0)
hip = C.CDLL("libamdhip64.so.7")
def free():
    a, b = C.c_size_t(), C.c_size_t()
    assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value
hs = rt.HostScene.workload(2, width=1920, height=1080, detail=12, n_spheres=16)
ds = rt.DeviceScene(hs)
kw = dict(mode=int(sys.argv[1]), max_level=int(sys.argv[2]))
ds.render(rt.params(64, 64, **kw), ids=False, tprim=False)
before = free()
ds.render(rt.params(1920, 1080, **kw), ids=False, tprim=False)
print("bytes", before - free())
"""


@pytest.mark.parametrize("mode,depth,per_sample", [
    (0x3, 0, HIT + COLOUR),  # a view: hits, no nodes
    (0x6, 0, HIT + NODE + MASK + 4 * SHADOW + COLOUR),
    (0x80, 4, 5 * (HIT + NODE + MASK + 4 * SHADOW) + 4 * RAY + COLOUR),  # rays that do not branch: no child slots
], ids=["normal view", "shadow view", "frame"])
def test_frame_takes_what_its_kernels_read(rt_gpu, mode, depth, per_sample):
    log(f"case: mode {mode:#x}, depth {depth}, {per_sample} bytes a sample")
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(mode), str(depth)], cwd=ROOT, capture_output=True, text=True,
                       timeout=60, env=os.environ)
    assert r.returncode == 0, r.stderr[-2000:]
    taken = int(r.stdout.split("bytes")[1].split()[0])
    # buffers are taken with a quarter of headroom; the frame's RGB comes on top,
    # and each of the buffers (six a level, and two) may round up to 2 MB
    most = SAMPLES * (per_sample * 5 / 4 + 3) + (6 * (depth + 1) + 2) * (2 << 20)
    log(f"  {taken / 1e6:.0f} MB of at most {most / 1e6:.0f} MB")
    assert 0 < taken <= most
