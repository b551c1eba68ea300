"""Short queues are walked with four lanes per ray, longer ones with one
(rt_quad.hpp): frames whose levels lie on both sides of the limit, and at the
edges of a wave of 16 rays, must equal the megakernel's, which always walks
one ray per lane, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import log

pytestmark = pytest.mark.gpu

LIMIT = 98304  # rays of a level, 256 CUs


def _scene(rt, name):
    if name == "refracting spheres":  # planes outside the BVH, self re-hits, two children
        hs = rt.HostScene.workload(1)
        for k in range(1, 5):
            hs.set_material(k, (0.1, 0.1, 0.1), (0.3, 0.4, 0.5), (0.5, 0.5, 0.5), 20.0, reflect=0.2, refract=0.6, rfr=1.4)
        return hs, 4
    if name == "soup":
        return rt.HostScene.workload(3, index=0, detail=20000), 4
    return rt.HostScene.workload(5, width=256, height=144, detail=32, n_spheres=24, n_lights=16), 5


@pytest.mark.parametrize("scene", ["refracting spheres", "soup", "terrain"])
@pytest.mark.parametrize("size", [(1, 1), (17, 3), (97, 61), (384, 256), (392, 256)],
                         ids=["1x1", "17x3", "97x61", "at_limit", "above_limit"])
def test_quads_equal_single_lanes(rt_gpu, scene, size):
    rt = rt_gpu
    hs, depth = _scene(rt, scene)
    ds = rt.DeviceScene(hs)
    W, H = size
    if size == (384, 256):
        assert W * H == LIMIT
    log(f"case: {scene} at {W}x{H}, depth {depth}")
    frame = lambda engine: ds.render(rt.params(W, H, max_level=depth, engine=engine))
    got, ref = frame(rt.RTG_ENGINE_WAVEFRONT), frame(rt.RTG_ENGINE_MEGAKERNEL)
    for k in ("rgb", "ids", "t"):
        assert np.array_equal(got[k], ref[k]), f"{k} differs"
    assert got["stats"].rays_total == ref["stats"].rays_total
