"""Scenes built into the device blocks that destroyed and replaced scenes leave:
frames of each must not depend on what its blocks held before, frames still on
a caller's stream when their scene is destroyed must be complete, and scenes
loaded on one thread must not disturb frames copied out on another (the
library's host threads serve both)."""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

from conftest import compare_frames, log
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

W, H = 160, 96


def _host(rt, seed, index=0, detail=9000):
    return rt.HostScene.workload(3, seed=seed, index=index, detail=detail, n_lights=2)


def test_recycled_blocks(rt_gpu):
    rt = rt_gpu
    p = rt.params(W, H, max_level=2)
    for k in range(4):  # the same sizes, another scene each time; a smaller one between
        hs = _host(rt, 1 + k, index=k % 2, detail=9000 - 900 * (k % 2))
        log(f"case: scene {k}, built, moved and refitted, rebuilt")
        ds = rt.DeviceScene(hs)
        for step in ("built", "moved", "rebuilt"):
            if step == "moved":
                hs.set_position(0, (0.5, -0.25, 0.75, 1.0))
                ds.update(hs)
            elif step == "rebuilt":
                ds.rebuild(hs)
            c = compare_frames(ds.render(p), po.OracleScene(hs.desc_ptr).render(p, po.ORACLE_REF32, threads=8))
            assert c["ids_mismatch_outside_band"] == 0 and c["rgb_over_1"] == 0, (step, c)
        ds.close()


def test_frames_in_flight_when_their_scene_is_destroyed(rt_gpu):
    rt = rt_gpu
    lib = rt._capi.load()
    hip = C.CDLL("libamdhip64.so.7")  # the runtime librtg loaded
    p = rt.params(1024, 768, max_level=3)
    stream, out = C.c_void_p(), [C.c_void_p() for _ in range(3)]
    size = 1024 * 768 * 3
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    for o in out:
        assert hip.hipMalloc(C.byref(o), C.c_size_t(size)) == 0
    want = rt.DeviceScene(_host(rt, 1)).render(p, ids=False, tprim=False)["rgb"]
    log("case: three frames on a caller's stream, their scene destroyed, another built in its blocks")
    ds = rt.DeviceScene(_host(rt, 1))
    for o in out:
        assert lib.rtg_render_device(ds.h, C.byref(p), o, None, None, None, stream) == 0
    ds.close()
    other = rt.DeviceScene(_host(rt, 2))
    got = np.empty((768, 1024, 3), np.uint8)
    assert hip.hipStreamSynchronize(stream) == 0
    for o in out:
        assert hip.hipMemcpy(got.ctypes.data_as(C.c_void_p), o, C.c_size_t(size), 2) == 0
        assert np.array_equal(got, want)
        assert hip.hipFree(o) == 0
    assert not np.array_equal(other.render(p, ids=False, tprim=False)["rgb"], want)
    assert hip.hipStreamDestroy(stream) == 0


def test_two_threads_share_the_host_threads(rt_gpu):
    rt = rt_gpu
    p = rt.params(1024, 768, max_level=1)
    ds = rt.DeviceScene(_host(rt, 3))
    want = ds.render(p)
    hs = rt.HostScene.workload(2, width=64, height=64, detail=60)
    small = rt.params(64, 64, max_level=1)
    want_small = rt.DeviceScene(hs).render(small)["rgb"]
    log("case: 12 scenes loaded, updated and rendered on one thread beside 24 frames on another")
    wrong = []

    def load():
        for _ in range(12):
            d = rt.DeviceScene(hs)
            d.update(hs)
            if d.stats()["shading_updates"] != 1 or not np.array_equal(d.render(small)["rgb"], want_small):
                wrong.append("loaded scene")
            d.close()

    def frames():
        for _ in range(24):
            got = ds.render(p)
            if not all(np.array_equal(got[k], want[k]) for k in ("rgb", "ids", "t")):
                wrong.append("frame")

    threads = [threading.Thread(target=f) for f in (load, frames)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
