"""The boxes of the radix tree's nodes are joined a block of 512 sorted
primitives at a time, and across blocks for the nodes that span them
(k_refit, k_refit_wide): scenes of sizes around whole blocks, built and
refitted after a move, against the oracle's scan of every object."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import compare_frames, log
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 64, 511, 512, 513, 1024, 1025, 4097])
def test_trees_around_whole_blocks(rt_gpu, n):
    rt = rt_gpu
    hs = rt.HostScene.workload(3, index=0, detail=n, n_lights=2)
    ds = rt.DeviceScene(hs)
    p = rt.params(96, 64, max_level=2)
    for move in (None, (0.75, -0.5, 1.25, 1.0)):
        if move is not None:
            hs.set_position(0, move)
            ds.update(hs)
            assert ds.stats()["refits"] == 1
        log(f"case: {n} triangles, {'moved and refitted' if move else 'built'}")
        ref = po.OracleScene(hs.desc_ptr).render(p, po.ORACLE_REF32, threads=4)
        c = compare_frames(ds.render(p), ref)
        assert c["ids_mismatch_outside_band"] == 0 and c["rgb_over_1"] == 0, c
        assert (ref["ids"] >= 0).any()
