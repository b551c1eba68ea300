"""Batches whose levels do not run as one launch each (k_step): those past its
longest (2^24 samples), which run on one stream, those with an FP64 re-test, and
those whose queues are sized by read-backs.  The shadow rays of these two run on
the side stream beside the next level, or with RTG_FLAG_ONE_STREAM on the
batch's own.  All must give each request's frame rendered alone, launched and
replayed from a graph."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import log

pytestmark = pytest.mark.gpu


def _items(rt, what):
    soup, spheres = rt.HostScene.workload(3, index=0, detail=20000), rt.HostScene.workload(1)
    ds = [rt.DeviceScene(soup), rt.DeviceScene(spheres)]
    if what == "long":
        assert 3 * 1600 * 1000 * 4 > 1 << 24
        return [(ds[k % 2], dict(width=1600, height=1000, max_level=2, spp=4, seed=k)) for k in range(3)], 0
    shapes = [(128, 64), (97, 80), (200, 121), (64, 64), (33, 47), (160, 96), (64, 128), (256, 64)]
    if what == "re-test":
        return [(ds[k % 2], dict(width=w, height=h, max_level=3, seed=k)) for k, (w, h) in enumerate(shapes)], \
            rt.RTG_FLAG_FP64_RETEST
    ds[1] = rt.DeviceScene(rt.HostScene.workload(5, width=256, height=144, detail=32, n_spheres=24, n_lights=16))
    # depth 15: two children a hit, 4 samples: a bound past any budget
    return [(ds[k % 2], dict(width=w, height=h, max_level=[3, 15][k % 2], spp=4, seed=k))
            for k, (w, h) in enumerate(shapes)], 0


@pytest.mark.parametrize("what,graph", [("long", True), ("re-test", True), ("read back", False)])
def test_unfused_batches_identical_on_one_stream(rt_gpu, what, graph):
    rt = rt_gpu
    items, flag = _items(rt, what)
    refs = [d.render(rt.params(**p, flags=flag), tprim=False) for d, p in items]
    for streams in (0, rt.RTG_FLAG_ONE_STREAM):
        batch = [(d, rt.params(**p, flags=flag | streams)) for d, p in items]
        log(f"case: {what} batch of {len(batch)}, {'one stream' if streams else 'side stream'}: eager, then 3 times")
        runs = [rt.render_batch(batch, eager=True)] + [rt.render_batch(batch) for _ in range(3)]
        assert runs[-1][1].graph_replays == (1 if graph else 0)
        for outs, st in runs:
            for o, ref in zip(outs, refs):
                assert np.array_equal(o["rgb"], ref["rgb"]) and np.array_equal(o["ids"], ref["ids"])
            assert st.rays_total == sum(x["stats"].rays_total for x in refs)
