"""Rays that hit their own analytic sphere again from inside take a second pass
through the walk (child_src): a scene of refracting spheres, a BallPlane and a
plane whose tree does not lie in LDS whole, at sizes on both sides of the limits
of four, sixteen and 64 rays to a wave, and in a batch, whose deeper levels are
k_step's.  Equal to the megakernel bit for bit, and at one size to the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import compare_frames, log
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

SIZES = [(64, 64), (65, 64), (384, 256), (392, 256)]  # 4,096 and 98,304 rays: the limits on 256 CUs
DEPTH = 5


@pytest.fixture(scope="module")
def scene(rt_gpu):
    rt = rt_gpu
    g = np.random.default_rng(11)
    hs = rt.HostScene.new()
    hs.set_env_light((0.1, 0.1, 0.1, 1.0))
    hs.add_plane()
    glass = dict(reflect=0.25, refract=0.6, rfr=1.4)
    for _ in range(300):  # overlapping: a ray inside one enters others
        s = hs.add_sphere(float(g.uniform(0.4, 1.0)))
        hs.set_position(s, (*g.uniform((-4, 1, -4), (4, 7, 4)).tolist(), 1.0))
        hs.set_material(s, (0.1, 0.1, 0.1), g.uniform(0.2, 0.9, 3).tolist(), (0.4, 0.4, 0.4), 24.0, **glass)
    b = hs.add_ballplane(0.5)
    hs.set_material(b, (0.1, 0.1, 0.1), (0.5, 0.6, 0.4), (0.4, 0.4, 0.4), 24.0, **glass)
    for p in ((6.0, 9.0, 8.0, 1.0), (-7.0, 6.0, 5.0, 1.0)):
        hs.set_light_position(hs.add_light(2, (0.2, 0.6, 0.3), (0.0, 0.0, 1.0, 256.0)), p)
    ds = rt.DeviceScene(hs)
    assert ds.stats()["n_nodes"] > 31  # else every level is walked lane by lane
    return hs, ds


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "%dx%d" % s)
def test_frames_equal_single_rays(rt_gpu, scene, size):
    rt, (hs, ds) = rt_gpu, scene
    log(f"case: {size[0]}x{size[1]}, depth {DEPTH}")
    frame = lambda engine: ds.render(rt.params(*size, max_level=DEPTH, engine=engine))
    got, ref = frame(rt.RTG_ENGINE_WAVEFRONT), frame(rt.RTG_ENGINE_MEGAKERNEL)
    for k in ("rgb", "ids", "t"):
        assert np.array_equal(got[k], ref[k]), f"{k} differs"
    a, b = got["stats"], ref["stats"]
    assert (a.rays_total, a.rays_refract) == (b.rays_total, b.rays_refract) and a.rays_refract > 0
    if size == SIZES[0]:
        c = compare_frames(got, po.OracleScene(hs.desc_ptr).render(rt.params(*size, max_level=DEPTH), po.ORACLE_REF32, threads=8))
        assert c["ids_mismatch_outside_band"] == 0 and c["rgb_over_1"] == 0, c


def test_batch_equals_single_rays(rt_gpu, scene):
    rt, (hs, ds) = rt_gpu, scene
    other = rt.DeviceScene(rt.HostScene.workload(3, index=0, detail=20000))
    items = [((ds, other)[k % 2], dict(width=w, height=h, max_level=DEPTH, seed=k))
             for k, (w, h) in enumerate(SIZES + [(33, 17), (97, 61)])]
    log(f"case: batch of {len(items)}")
    outs, _ = rt.render_batch([(d, rt.params(**p)) for d, p in items])
    for (d, p), o in zip(items, outs):
        ref = d.render(rt.params(**p, engine=rt.RTG_ENGINE_MEGAKERNEL))
        assert np.array_equal(o["rgb"], ref["rgb"]) and np.array_equal(o["ids"], ref["ids"])
