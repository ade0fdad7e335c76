"""The hand-over of counts between the workgroups of a one-launch pass: passes whose tiles publish at once (nothing in
view: no load of theirs is used before) and passes of few and of many tiles, unwaited on one stream, bit-exact against
the oracle. Needs a GPU."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz
from oracle import pyoracle as orc
from tests import helpers as H

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
