"""The cluster cull around the number of object tiles whose expansion writes its own draws (640 tiles of 1024 objects),
and tiles whose records take one chunk of a workgroup and several; each after ascending, unordered and repeated transform
updates; bit-exact against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import cull as bz
from oracle import pyoracle as orc
from tests import helpers as H
from tests.test_gpu_cluster import ALL, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1023, 1025, 30000, 640 * 1024, 640 * 1024 + 1])
@pytest.mark.parametrize("order", ["ascending", "shuffled", "repeated"])
def test_cluster_tiles(n, order):
    sc = bz.synth_scene(40 + n, n, 64, 4, clusters=(16, 64))
    rng = np.random.default_rng(n)
    xfs = sc.transforms.copy()
    # a third of the objects in front of the camera: several chunks of records in some tiles
    near = np.arange(n) % 4096 < 1400
    xfs["pos"][near] = np.stack([rng.uniform(-20, 20, n), rng.uniform(-10, 10, n), rng.uniform(20, 90, n)],
                                1).astype(np.float32)[near]
    v = H.view(pyr=(512, 256))
    with bz.Context(0) as ctx:
        h = ctx.scene_create(sc.objects, xfs, sc.surfaces, sc.lods)
        ctx.scene_set_clusters(h, sc.clusters)
        depth = bz.synth_depth(9, 1024, 512, 60, v.proj5, 0.1)
        buf = ctx.alloc(depth.nbytes)
        buf.upload(depth)
        pyr = ctx.pyramid_create(512, 256, 9)
        ctx.pyramid_build(pyr, buf.ptr, 1024, 512)
        ids = np.unique(rng.integers(0, n, max(1, n // 50), dtype=np.uint32))
        if order == "shuffled":
            rng.shuffle(ids)
        elif order == "repeated":
            ids = np.concatenate([ids, ids[::-1], ids[:1]])
        new = xfs[ids].copy()
        new["pos"] += rng.uniform(-5, 5, (len(ids), 3)).astype(np.float32)
        for k, i in enumerate(ids):  # the last occurrence of an id wins
            xfs[i] = new[k]
        ctx.update_transforms(h, ids, new)
        opyr = orc.pyramid(orc.pyramid_build(depth, 512, 256, 9), 512, 256, 9)
        cap = 1 << 22
        recs, nd, cmds, nc = run_oracle(sc, v, ALL, opyr, dcap=cap, cap=cap, transforms=xfs)
        assert nd <= cap
        for _ in range(2):  # the second call's published counts are not the first one's
            got = run_gpu(ctx, h, v, ALL, pyr, dcap=cap, cap=cap)
            assert (got[1], got[3]) == (nd, nc)
            assert np.array_equal(got[0], recs)
            assert np.array_equal(got[2], cmds)
