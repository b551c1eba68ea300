"""Walks whose stack outgrows the LDS of four lanes (52 entries of QuadStack): a
tree with a chain of 30 levels, one for each bit of the Morton code, above
spheres that share the code 0.  Seen from beyond them every box of the chain is
met, the deep end first, so that a walk leaves three entries a level on its way.
Four rays, sixteen rays and 64 rays to a wave, against the megakernel and the
oracle's scan of every object."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import compare_frames, emul_render, log
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

EXTENT = 4.0   # of the sphere centres, 1024 Morton cells
N_DEEP = 2048  # spheres in the cell of code 0


class _Seen:
    """The scene with its camera on the diagonal, looking at the origin."""

    def __init__(self, rt, hs):
        self.keep = hs
        self.desc = rt._capi.rtg_scene_desc.from_buffer_copy(C.string_at(hs.desc_ptr, C.sizeof(rt._capi.rtg_scene_desc)))
        r = lambda v: rt._capi.rtg_vec4(*(np.asarray(v, np.float64) / np.linalg.norm(v)).tolist(), 0.0)
        cam = self.desc.camera
        cam.position = rt._capi.rtg_vec4(-8.0, -8.0, -8.0, 1.0)
        cam.n, cam.u, cam.v = r((1, 1, 1)), r((1, 0, -1)), r((-1, 2, -1))
        self.desc_ptr = C.addressof(self.desc)


def _scene(rt):
    hs = rt.HostScene.new()
    hs.set_env_light((0.1, 0.1, 0.1, 1.0))
    put = lambda r, at: hs.set_position(hs.add_sphere(float(r)), (*(float(x) for x in at), 1.0))
    for r in np.random.default_rng(3).permutation(np.linspace(2.6, 3.0, N_DEEP)):
        put(r, (0, 0, 0))  # entered first from the camera's side: the largest
    for bit in range(10):
        for axis in range(3):
            at = np.zeros(3)
            at[axis] = (2**bit + 0.5) / 1024 * EXTENT
            for k in range(4):  # more than a leaf holds
                put(2.5 - 0.01 * k, at)
    put(0.1, (EXTENT, 0, 0))  # the extent of the Morton grid
    light = hs.add_light(2, (0.2, 0.6, 0.3), (0.0, 0.0, 1.0, 256.0))
    hs.set_light_position(light, (-9.0, -6.0, -8.0, 1.0))
    return _Seen(rt, hs)


@pytest.mark.parametrize("size", [(61, 37), (97, 61), (392, 256)], ids=["four rays", "sixteen rays", "64 rays"])
def test_stack_past_the_lds_of_four_lanes(rt_gpu, size):
    rt = rt_gpu
    hs = _scene(rt)
    p = rt.params(*size, max_level=1)
    small = rt.params(61, 37, max_level=1)
    deepest = emul_render(hs.desc_ptr, small)["max_stack"]
    log(f"case: {size[0]}x{size[1]}, {deepest} stack entries")
    assert 52 < deepest <= 96
    ds = rt.DeviceScene(hs)
    got = ds.render(p)
    ref = ds.render(rt.params(*size, max_level=1, engine=rt.RTG_ENGINE_MEGAKERNEL))
    for k in ("rgb", "ids", "t"):
        assert np.array_equal(got[k], ref[k]), f"{k} differs"
    if size[0] < 100:
        o = po.OracleScene(hs.desc_ptr).render(p, po.ORACLE_REF32, threads=8)
        c = compare_frames(got, o)
        assert c["ids_mismatch_outside_band"] == 0 and c["rgb_over_1"] == 0, c
        assert (o["ids"] >= 0).any()
