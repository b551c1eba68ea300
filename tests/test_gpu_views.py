"""The primary-only modes (depth, normal, texture, material and shadow test,
RayTracer.cpp:46-330) on both engines: the wavefront's k_extend and k_view, and
the megakernel, whose samples walk one ray per lane.  Equal bit for bit, on
trees past the ones that lie in LDS whole, and with the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import compare_frames, log
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

MODES = [0x2, 0x3, 0x4, 0x5, 0x6]


def _both(rt, ds, W, H, **kw):
    got, ref = (ds.render(rt.params(W, H, engine=e, **kw)) for e in (rt.RTG_ENGINE_WAVEFRONT, rt.RTG_ENGINE_MEGAKERNEL))
    for k in ("rgb", "ids", "t"):
        assert np.array_equal(got[k], ref[k]), f"{k} differs"
    a, b = got["stats"], ref["stats"]
    assert (a.rays_primary, a.rays_shadow, a.rays_total) == (b.rays_primary, b.rays_shadow, b.rays_total)
    return got


@pytest.fixture(scope="module")
def mesh(rt_gpu):
    hs = rt_gpu.HostScene.workload(2, width=211, height=133, detail=20)
    ds = rt_gpu.DeviceScene(hs)
    assert ds.stats()["n_nodes"] > 31
    return hs, ds


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("options", [dict(), dict(spp=4, seed=3), dict(tile_compat=1), dict(max_level=5)],
                         ids=["plain", "4 samples", "tiles", "depth ignored"])
def test_engines_agree(rt_gpu, mesh, mode, options):
    hs, ds = mesh
    log(f"case: mode {mode:#x}, 211x133, {options}")
    kw = {"max_level": 0, **options}
    got = _both(rt_gpu, ds, 211, 133, mode=mode, **kw)
    if options == {}:
        ref = po.OracleScene(hs.desc_ptr).render(rt_gpu.params(211, 133, mode=mode, max_level=0), po.ORACLE_REF32, threads=8)
        c = compare_frames(got, ref)
        assert c["ids_mismatch_outside_band"] == 0 and c["rgb_over_1"] == 0, c


@pytest.mark.parametrize("mode", MODES)
def test_engines_agree_without_lights(rt_gpu, mode):
    rt = rt_gpu
    hs = rt.HostScene.workload(2, width=97, height=61, detail=10, n_lights=2)
    for k in range(2):
        hs.switch(1, k, False)  # Scene::Switch of a light
    log(f"case: mode {mode:#x}, 97x61, no light on")
    got = _both(rt, rt.DeviceScene(hs), 97, 61, mode=mode, max_level=0)
    assert got["stats"].rays_shadow == 0


@pytest.mark.parametrize("mode", [0x3, 0x6])
def test_engines_agree_over_several_passes(rt_gpu, mesh, mode):
    W, H = 2048, 520
    assert W * H * 4 > 1 << 22  # more samples than a pass holds
    log(f"case: mode {mode:#x}, {W}x{H} at 4 samples, two passes")
    _both(rt_gpu, mesh[1], W, H, mode=mode, max_level=0, spp=4, seed=1)
