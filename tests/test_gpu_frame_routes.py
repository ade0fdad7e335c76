"""Frame-cache passes on routes that other tests do not reach: recording EARLY and cached LATE whose emit reads a scan of the
tile counts (just over 32 768 tiles), and tiles of 1024 recorded objects in a 256-thread decide, most of them survivors;
bit-exact against the oracle. Needs a GPU."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz
from oracle import pyoracle as orc
from tests import helpers as H
from tests import test_gpu_frame_cache as FCT

pytestmark = pytest.mark.gpu

ctx, pyramid = FCT.ctx, FCT.pyramid


def test_dense_survivors_four_items(ctx, pyramid):
    FCT.test_frame_cache_dense_survivors(ctx, pyramid, (256, 4))


def test_frame_behind_a_scan(ctx, pyramid):
    n = 32768 * 512 + 1
    sc = H.c1_scene(n)
    scene = H.as_tuple(sc)
    p, opyr = pyramid
    v = H.view(pyr=(1024, 512))
    vb, cap = H.view_bytes(v), n // 4
    vis0 = bz.synth_visibility(H.SEED_C1, n, 0.5)
    h = ctx.scene_create(*scene)
    old = ctx.get_tuning(0)
    cmds, cnt = ctx.alloc(cap * 24), ctx.alloc(4)
    try:
        ctx.set_tuning(0, 256, 2, 8)  # tiles of 512 objects
        ctx.set_visibility(h, vis0)
        for pass_ in (A.PASS_EARLY, A.PASS_LATE):
            ctx.cull(h, v, pass_, cmds, cnt, capacity=cap, pyramid=p, flags=A.CULL_FRAME_CACHE)
            ctx.check_kernels()
            got, total = ctx.read_commands(cmds, cnt, capacity=cap)
            vexp = vis0.copy()
            late = pass_ == A.PASS_LATE
            exp, ne = orc.cull(scene, vb, pass_, opyr if late else None, vis_in=vexp, vis_out=vexp if late else None,
                               capacity=cap, threads=16)
            assert total == ne and total > 0
            np.testing.assert_array_equal(H.cmds_u32(got), exp)
        np.testing.assert_array_equal(ctx.get_visibility(h, n), vexp)
        assert ctx.frame_cache_stats(h) == (1, 1)
    finally:
        ctx.set_tuning(0, old.block, old.items, old.grid_per_cu, old.reserved)
        cmds.free()
        cnt.free()
        ctx.scene_destroy(h)
