"""Batches around the number of jobs that travel in the kernel arguments (12 views, 16 pyramids): eager, twice in a row
without waiting, and replayed from a graph, each view bit-exact against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz
from tests import helpers as H
from tests.test_gpu_batch import Job, oracle_pyramid

pytestmark = pytest.mark.gpu

PASSES = [A.PASS_LATE, A.PASS_PLAIN, A.PASS_TEMPORAL]


@pytest.mark.parametrize("views", [1, 2, 11, 12, 13, 16, 17, 18])
@pytest.mark.parametrize("graph", [False, True])
def test_few_jobs(views, graph):
    """Ranges of 1 to 3000 objects (tiles of one job and of many, jobs that end inside an emit workgroup's tiles), every
    third job without a pyramid, one without objects."""
    ctx = bz.Context(0)
    try:
        sc = H.as_tuple(H.c1_scene(20000, seed=views))
        h = ctx.scene_create(*sc)
        rng = np.random.default_rng(views)
        jobs, builds, pyramids = [], [], []
        for k in range(views):
            w, hh = (256, 256) if k % 2 else (300, 200)
            bw, bh, mips = (128, 128, 7)
            buf = ctx.alloc(w * hh * 4)
            ctx.synth_depth_device(7 + k, w, hh, 20, H.view(w=w, h=hh).proj5, 0.1, buf.ptr)
            p = ctx.pyramid_create(bw, bh, mips)
            builds.append((p, buf.ptr, w, hh))
            pyramids.append((p, buf, bw, bh, mips, w, hh))
            v = H.view(fov=60 + k, w=w, h=hh, yaw=0.3 * k, pyr=(bw, bh))
            pass_ = PASSES[k % 3]
            n = int(rng.integers(1, 3001)) if k else 1
            jobs.append(Job(ctx, h, sc, v, pass_, pyr=None if pass_ == A.PASS_PLAIN else pyramids[k],
                            begin=int(rng.integers(1, 20000 - n)), count=n, seed=k))
        empty = Job(ctx, h, sc, H.view(), A.PASS_PLAIN, begin=5, count=0)
        table = [j.vj for j in jobs[:1]] + [empty.vj] + [j.vj for j in jobs[1:]]
        ctx.sync()
        if graph:
            g = ctx.batch_graph_create(builds, table)
            for _ in range(3):
                ctx.graph_launch(g)
                ctx.check_kernels()
        else:
            for _ in range(2):
                ctx.pyramid_build_batch(builds)
                ctx.cull_batch(table)
        ctx.check_kernels()
        assert int(empty.cnt.download(np.uint32, 1)[0]) == 0
        for j, (p, buf, bw, bh, mips, w, hh) in zip(jobs, pyramids):
            j.check(ctx, None if j.pyr is None else oracle_pyramid(buf, bw, bh, mips, w, hh))
    finally:
        ctx.close()


def test_table_grows_behind_a_running_batch():
    """A batch of large jobs, and without waiting for it one of far more jobs, whose table has to grow."""
    ctx = bz.Context(0)
    try:
        n = 600000
        sc = H.as_tuple(H.c1_scene(n, seed=3))
        h = ctx.scene_create(*sc)
        s = ctx.stream()
        large = [Job(ctx, h, sc, H.view(yaw=0.3 * k), A.PASS_PLAIN, begin=0, count=n) for k in range(13)]
        small = [Job(ctx, h, sc, H.view(yaw=0.01 * k), A.PASS_PLAIN, begin=11 * k, count=300 + k) for k in range(300)]
        ctx.sync()
        for jobs in (large, small):
            ctx.cull_batch([j.vj for j in jobs], stream=s)
        ctx.check_kernels(s)
        for j in large[::4] + small[::29]:
            j.check(ctx, None)
    finally:
        ctx.close()
