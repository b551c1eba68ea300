"""The walks of a level (rtg_wave.hip, Walk): lane by lane where a level is
known to hold 2^20 rays or the tree lies in LDS whole, else the wave's rays
together, whose last 16 go on with four lanes each and whose idle lanes take
subtrees over (rt_quad.hpp); four rays to a wave up to 4096.  Around the limits, and with a few slow rays among
quick ones, frames must equal the megakernel's, which always walks one ray per
lane on its own, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import log

pytestmark = pytest.mark.gpu


def _spheres(rt, n):
    """n spheres on a spiral, with two lights; the tree's 4-wide nodes grow with n."""
    hs = rt.HostScene.new()
    hs.set_env_light((0.1, 0.1, 0.1, 1.0))
    hs.add_plane()
    for k in range(n):
        a = 2.4 * k
        s = hs.add_sphere(0.5)
        hs.set_position(s, (0.03 * k * np.cos(a), 1.0 + 0.01 * k, 0.03 * k * np.sin(a), 1.0))
        hs.set_material(s, (0.1, 0.1, 0.1), (0.3, 0.4, 0.5), (0.5, 0.5, 0.5), 20.0, reflect=0.4)
    for p in ((6.0, 9.0, 8.0, 1.0), (-7.0, 6.0, 5.0, 1.0)):
        hs.set_light_position(hs.add_light(2, (0.2, 0.6, 0.3), (0.0, 0.0, 1.0, 256.0)), p)
    return hs


@pytest.mark.parametrize("scene,size", [
    ("spheres 0", (97, 61)), ("spheres 1", (97, 61)), ("spheres 3", (97, 61)), ("spheres 30", (200, 133)),
    ("spheres 130", (200, 133)), ("spheres 600", (1024, 1023)), ("soup", (1024, 1023)), ("soup", (1024, 1024)),
    ("field", (640, 401)), ("soup", (64, 64)), ("soup", (65, 64)), ("field", (64, 60))], ids=lambda v: v if isinstance(v, str) else "%dx%d" % v)
def test_walks_equal_single_rays(rt_gpu, scene, size):
    rt = rt_gpu
    if scene.startswith("spheres"):
        hs = _spheres(rt, int(scene.split()[1]))
    else:  # rays along the grain of a height field are slow, most others quick
        hs = rt.HostScene.workload(3, index=0 if scene == "soup" else 1, detail=30000, n_lights=2)
    ds = rt.DeviceScene(hs)
    log(f"case: {scene} at {size[0]}x{size[1]}")
    frame = lambda engine: ds.render(rt.params(*size, max_level=3, engine=engine))
    got, ref = frame(rt.RTG_ENGINE_WAVEFRONT), frame(rt.RTG_ENGINE_MEGAKERNEL)
    for k in ("rgb", "ids", "t"):
        assert np.array_equal(got[k], ref[k]), f"{k} differs"
    assert got["stats"].rays_total == ref["stats"].rays_total
