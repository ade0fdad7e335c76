"""Passes over few objects run in one launch (up to 327 680 objects, tiles of 512): every pass at the edges of the tiles
and of that range, in turn on one stream, on ranges and visibility buffers of any alignment, and replayed from a graph
between eager passes; bit-exact against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz
from blitzen_amd.hip import StreamGraph
from oracle import pyoracle as orc
from tests import helpers as H

pytestmark = pytest.mark.gpu

W, HH, BW, BH, MIPS = 640, 360, 512, 256, 9
MOST = 327680


@pytest.fixture(scope="module")
def world():
    """A scene in region order (all of a tile in view, or none of it) and a pyramid of its view."""
    ctx = bz.Context(0)
    n = MOST + 2000
    sc = bz.synth_scene(77, n, 256, 8)
    order = np.lexsort((sc.transforms["pos"][:, 0] // 40, sc.transforms["pos"][:, 2] // 40))
    sc.transforms = np.ascontiguousarray(sc.transforms[order])
    v = H.view(fov=80, w=W, h=HH, pyr=(BW, BH))
    depth = bz.synth_depth(5, W, HH, 40, v.proj5, 0.1)
    buf = ctx.alloc(depth.nbytes)
    buf.upload(depth)
    pyr = ctx.pyramid_create(BW, BH, MIPS)
    ctx.pyramid_build(pyr, buf.ptr, W, HH)
    vis = bz.synth_visibility(3, n, 0.4)
    state = {"ctx": ctx, "scene": H.as_tuple(sc), "h": ctx.scene_create(*H.as_tuple(sc)), "view": v, "pyr": pyr,
             "opyr": orc.pyramid(orc.pyramid_build(depth, BW, BH, MIPS), BW, BH, MIPS), "vis": vis, "n": n,
             "cmds": ctx.alloc(n * 24), "cnt": ctx.alloc(4), "vin": ctx.alloc(n * 4), "vout": ctx.alloc(n * 4)}
    state["vin"].upload(vis)
    yield state
    ctx.close()


def run(w, pass_, begin, n, flags=0, capacity=None, stream=None):
    late = pass_ == A.PASS_LATE
    w["ctx"].cull(w["h"], w["view"], pass_, w["cmds"], w["cnt"], capacity=w["n"] if capacity is None else capacity,
                  pyramid=w["pyr"] if pass_ != A.PASS_PLAIN else 0, flags=flags, begin=begin, n=n,
                  vis_in=w["vin"].ptr if late or pass_ == A.PASS_EARLY else None, vis_out=w["vout"].ptr if late else None,
                  stream=stream)


def check(w, pass_, begin, n, capacity=None, stream=None):
    cap = w["n"] if capacity is None else capacity
    got, total = w["ctx"].read_commands(w["cmds"], w["cnt"], capacity=cap, stream=stream)
    vexp = np.full(w["n"], 7, np.uint32) if pass_ == A.PASS_LATE else None
    exp, ne = orc.cull(w["scene"], H.view_bytes(w["view"]), pass_, None if pass_ == A.PASS_PLAIN else w["opyr"],
                       begin=begin, count=n, vis_in=w["vis"], vis_out=vexp, capacity=cap, threads=8)
    assert total == ne, (pass_, begin, n, total, ne)
    np.testing.assert_array_equal(H.cmds_u32(got), exp)
    if vexp is not None:
        np.testing.assert_array_equal(w["vout"].download(np.uint32, w["n"], stream), vexp)


RANGES = [(0, 1), (3, 511), (0, 512), (1, 513), (7, 5000), (1024, 131072), (5, MOST - 1), (0, MOST), (2, MOST + 1)]


@pytest.mark.parametrize("begin,n", RANGES)
@pytest.mark.parametrize("pass_", [A.PASS_EARLY, A.PASS_LATE, A.PASS_PLAIN, A.PASS_TEMPORAL])
def test_passes(world, begin, n, pass_):
    world["vout"].fill_u32(7)
    run(world, pass_, begin, n)
    check(world, pass_, begin, n)


@pytest.mark.parametrize("begin,n", RANGES)
def test_frame_cache(world, begin, n):
    """EARLY records, LATE reads the records: the same results, also when nothing fits the command buffer."""
    world["vout"].fill_u32(7)
    run(world, A.PASS_EARLY, begin, n, flags=A.CULL_FRAME_CACHE)
    check(world, A.PASS_EARLY, begin, n)
    for capacity in (None, 0, 3):
        run(world, A.PASS_LATE, begin, n, flags=A.CULL_FRAME_CACHE, capacity=capacity)
        check(world, A.PASS_LATE, begin, n, capacity=capacity)


def test_many_sizes_on_one_stream(world):
    """Launches of many and of few tiles in turn, unwaited: no count of one launch is taken by another."""
    s = world["ctx"].stream()
    rng = np.random.default_rng(1)
    for _ in range(40):
        begin = int(rng.integers(0, 4000))
        run(world, A.PASS_PLAIN, begin, int(rng.choice([1, 600, 3000, 200000])), stream=s)
    for begin, n in ((11, 150001), (0, 700), (13, 300000)):
        run(world, A.PASS_TEMPORAL, begin, n, stream=s)
        check(world, A.PASS_TEMPORAL, begin, n, stream=s)
    world["ctx"].check_kernels(s)


def test_graph_replays_between_eager_passes(world):
    s = world["ctx"].stream()
    world["vout"].fill_u32(7)
    world["ctx"].sync()

    def frame():
        run(world, A.PASS_EARLY, 9, 100000, flags=A.CULL_FRAME_CACHE, stream=s)
        run(world, A.PASS_LATE, 9, 100000, flags=A.CULL_FRAME_CACHE, stream=s)

    frame()
    world["ctx"].sync(s)
    g = StreamGraph(s, frame)
    for k in range(4):
        run(world, A.PASS_PLAIN, 0, 1000 * (k + 1), stream=s)
        check(world, A.PASS_PLAIN, 0, 1000 * (k + 1), stream=s)
        g.launch(s)
        check(world, A.PASS_LATE, 9, 100000, stream=s)
    world["ctx"].check_kernels(s)


def test_first_call_on_a_captured_stream(world):
    """A stream's hand-off words are allocated by its first call, which is refused under capture; after one call outside,
    the same call is captured and replayed."""
    s = world["ctx"].stream()
    got = []

    def first():
        with pytest.raises(A.BzError) as e:
            run(world, A.PASS_PLAIN, 0, 3000, stream=s)
        got.append(e.value.status)

    StreamGraph(s, first)
    assert got == [A.E_STATE]
    run(world, A.PASS_PLAIN, 0, 3000, stream=s)
    check(world, A.PASS_PLAIN, 0, 3000, stream=s)
    g = StreamGraph(s, lambda: run(world, A.PASS_PLAIN, 5, 2000, stream=s))
    for _ in range(3):
        run(world, A.PASS_PLAIN, 0, 3000, stream=s)
        g.launch(s)
        check(world, A.PASS_PLAIN, 5, 2000, stream=s)
