"""The hand-over of counts between the workgroups of a one-launch pass: passes whose tiles publish at once (nothing in
view: no load of theirs is used before), of few and of many tiles, unwaited on one stream; tiles that do not wait for the
earlier ones' counts and leave their commands to the last tile (a wait limit of 0); and several streams at once; bit-exact
against the oracle. Needs a GPU."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz
from oracle import pyoracle as orc
from tests import helpers as H
from tests.test_gpu_cluster import run_oracle

pytestmark = pytest.mark.gpu

N, BW, BH, MIPS = 200_003, 512, 256, 9


@pytest.fixture(scope="module")
def world():
    ctx = bz.Context(0)
    sc = bz.synth_scene(78, N, 64, 4)
    depth = bz.synth_depth(6, 640, 360, 40, H.view(w=640, h=360).proj5, 0.1)
    buf = ctx.alloc(depth.nbytes)
    buf.upload(depth)
    pyr = ctx.pyramid_create(BW, BH, MIPS)
    ctx.pyramid_build(pyr, buf.ptr, 640, 360)
    vis = bz.synth_visibility(4, N, 0.4)
    w = {"ctx": ctx, "scene": H.as_tuple(sc), "h": ctx.scene_create(*H.as_tuple(sc)), "pyr": pyr, "vis": vis,
         "opyr": orc.pyramid(orc.pyramid_build(depth, BW, BH, MIPS), BW, BH, MIPS), "vin": ctx.alloc(N * 4),
         "vout": ctx.alloc(N * 4), "cmds": ctx.alloc(N * 24), "cnt": ctx.alloc(4),
         "in": H.view(fov=80, w=640, h=360, pyr=(BW, BH)),
         "out": H.view(fov=80, w=640, h=360, pos=(0.0, 0.0, 5000.0), pyr=(BW, BH))}
    w["vin"].upload(vis)
    ctx.sync()
    yield w
    ctx.close()


def frame(w, view, n, stream):
    for pass_ in (A.PASS_EARLY, A.PASS_LATE):
        w["ctx"].cull(w["h"], w[view], pass_, w["cmds"], w["cnt"], capacity=N, pyramid=w["pyr"],
                      flags=A.CULL_FRAME_CACHE, begin=0, n=n, vis_in=w["vin"].ptr, vis_out=w["vout"].ptr, stream=stream)


def check_late(w, view, n, stream):
    got, total = w["ctx"].read_commands(w["cmds"], w["cnt"], capacity=N, stream=stream)
    vexp = np.full(N, 7, np.uint32)
    exp, ne = orc.cull(w["scene"], H.view_bytes(w[view]), A.PASS_LATE, w["opyr"], begin=0, count=n, vis_in=w["vis"],
                       vis_out=vexp, capacity=N, threads=8)
    assert total == ne
    np.testing.assert_array_equal(H.cmds_u32(got), exp)
    np.testing.assert_array_equal(w["vout"].download(np.uint32, N, stream)[:n], vexp[:n])


@pytest.mark.parametrize("n", [512, 5000, N])
def test_tiles_that_publish_at_once(world, n):
    s = world["ctx"].stream()
    for k in range(30):
        frame(world, "out", (n, 1, N)[k % 3], s)
    frame(world, "out", n, s)
    check_late(world, "out", n, s)
    for k in range(10):
        frame(world, "out", n, s)
        frame(world, "in", n, s)
    check_late(world, "in", n, s)
    world["ctx"].check_kernels(s)


PASSES = [A.PASS_EARLY, A.PASS_LATE, A.PASS_PLAIN, A.PASS_TEMPORAL]


@pytest.mark.parametrize("limit", [0, 1, A.DEFAULT_WAIT_LIMIT])
@pytest.mark.parametrize("n", [513, 5000, N])
def test_commands_left_to_the_last_tile(world, limit, n):
    """With a wait limit of 0, a tile leaves its commands to the last one as soon as an earlier tile's count is not there:
    the results are the same, no wait is given up, and the launches after it are as usual."""
    w, ctx = world, world["ctx"]
    s = ctx.stream()
    try:
        ctx.set_wait_limit(limit)
        for capacity in (N, 100):
            for _ in range(3):
                for pass_ in PASSES:
                    ctx.cull(w["h"], w["in"], pass_, w["cmds"], w["cnt"], capacity=capacity,
                             pyramid=w["pyr"] if pass_ != A.PASS_PLAIN else 0, begin=0, n=n, vis_in=w["vin"].ptr,
                             vis_out=w["vout"].ptr, stream=s)
                    got, total = ctx.read_commands(w["cmds"], w["cnt"], capacity=capacity, stream=s)
                    vexp = np.full(N, 7, np.uint32) if pass_ == A.PASS_LATE else None
                    exp, ne = orc.cull(w["scene"], H.view_bytes(w["in"]), pass_, w["opyr"] if pass_ != A.PASS_PLAIN
                                       else None, begin=0, count=n, vis_in=w["vis"], vis_out=vexp, capacity=capacity,
                                       threads=8)
                    assert total == ne, (pass_, capacity)
                    np.testing.assert_array_equal(H.cmds_u32(got), exp)
            frame(w, "in", n, s)
            check_late(w, "in", n, s)
        ctx.check_kernels(s)
    finally:
        ctx.set_wait_limit(A.DEFAULT_WAIT_LIMIT)
    frame(w, "in", n, s)
    check_late(w, "in", n, s)


@pytest.mark.parametrize("limit", [0, A.DEFAULT_WAIT_LIMIT])
def test_cluster_culls_on_several_streams(limit):
    """Cluster culls of 640 and 300 tiles on five streams at once, all waiting among their own tiles, also with every tile
    leaving its draws at the first look; every stream's records and draws as the oracle's."""
    n = 640 * 1024
    sc = bz.synth_scene(51, n, 64, 4, clusters=(16, 64))
    rng = np.random.default_rng(51)
    near = np.arange(n) % 4096 < 200  # several chunks of draws in some tiles
    sc.transforms["pos"][near] = np.stack([rng.uniform(-20, 20, n), rng.uniform(-10, 10, n), rng.uniform(20, 90, n)],
                                          1).astype(np.float32)[near]
    v = H.view(pyr=(512, 256))
    with bz.Context(0) as ctx:
        ctx.set_wait_limit(limit)
        small, cap = 300 * 1024, 1 << 21
        scenes = []
        for m in (n, small):
            objs = (sc.objects[:m], sc.transforms[:m], sc.surfaces, sc.lods)
            h = ctx.scene_create(*objs)
            ctx.scene_set_clusters(h, sc.clusters)
            part = bz.SynthScene(*objs, sc.clusters)
            scenes.append((h, run_oracle(part, v, A.CLUSTER_FRUSTUM, dcap=cap, cap=cap)))
        runs = []
        for k in range(5):
            h, want = scenes[k & 1]
            out = [ctx.alloc(b) for b in (cap * 12, 4, cap * 24, 4)]
            runs.append((ctx.stream(), h, want, *out))
        ctx.sync()
        for _ in range(4):
            for s, h, _w, rec, nrec, cmds, cnt in runs:
                ctx.cull_clusters(h, v, A.CLUSTER_FRUSTUM, rec, nrec, cmds, cnt, dispatch_capacity=cap, capacity=cap,
                                  stream=s)
        for s, _h, (recs, nd, draws, nc), rec, nrec, cmds, cnt in runs:
            ctx.check_kernels(s)
            assert int(nrec.download(np.uint32, 1, s)[0]) == nd and int(cnt.download(np.uint32, 1, s)[0]) == nc
            np.testing.assert_array_equal(rec.download(np.uint32, nd * 3, s).reshape(-1, 3), recs)
            np.testing.assert_array_equal(cmds.download(np.uint32, nc * 6, s).reshape(-1, 6), draws)
