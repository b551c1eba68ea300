"""Walks whose stack outgrows its LDS part (16 entries a lane): spheres around
one centre, whose boxes every ray meets, so each level of the tree leaves three
entries.  Frames walked a lane per ray and four lanes per ray, against the
oracle's scan of every object."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import compare_frames, emul_render, log
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

N = 8192  # 12 internal levels of the radix tree, 6 four-wide ones: 18 entries


def _scene(rt):
    hs = rt.HostScene.new()
    hs.set_env_light((0.1, 0.1, 0.1, 1.0))
    r = np.random.default_rng(5).permutation(np.linspace(2.0, 3.0, N))
    for k in range(N):
        hs.set_position(hs.add_sphere(float(r[k])), (0.0, 4.0, 0.0, 1.0))
    light = hs.add_light(2, (0.2, 0.6, 0.3), (0.0, 0.0, 1.0, 256.0))
    hs.set_light_position(light, (6.0, 9.0, 8.0, 1.0))
    return hs


@pytest.mark.parametrize("size", [(61, 37), (392, 256)], ids=["four_lanes", "one_lane"])
def test_stack_past_its_lds_part(rt_gpu, size):
    rt = rt_gpu
    hs = _scene(rt)
    p = rt.params(*size, max_level=1)
    tiles = np.array([0 if size[0] < 64 else 17], np.int32)  # a tile the spheres cover
    e = emul_render(hs.desc_ptr, p, tiles=tiles)
    assert e["max_stack"] > 16
    log(f"case: {N} spheres at {size[0]}x{size[1]}, {e['max_stack']} stack entries")
    got = rt.DeviceScene(hs).render(p)
    ref = po.OracleScene(hs.desc_ptr).render(p, po.ORACLE_REF32, threads=8)
    c = compare_frames(got, ref)
    assert c["ids_mismatch_outside_band"] == 0 and c["rgb_over_1"] == 0, c
    assert (ref["ids"] >= 0).any()
