"""The emit's launch shapes by tile count: plain stores up to 4096 tiles, 16 tiles per workgroup and 16-byte stores above,
behind a scan above 32 768 tiles; at those edges, with truncated output, bit-exact against the oracle. Needs a GPU."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz
from oracle import pyoracle as orc
from tests import helpers as H

pytestmark = pytest.mark.gpu

TILE = 512
MOST = 32768 * TILE + 1


@pytest.fixture(scope="module")
def world():
    ctx = bz.Context(0)
    ctx.set_tuning(0, 256, 2, 8)  # tiles of 512 objects
    sc = H.as_tuple(H.c1_scene(MOST))
    h = ctx.scene_create(*sc)
    cmds, cnt = ctx.alloc((MOST // 4 + 1) * 24), ctx.alloc(4)
    yield ctx, sc, h, cmds, cnt
    ctx.close()


@pytest.mark.parametrize("begin,n", [(MOST - 4096 * TILE, 4096 * TILE), (3, 4096 * TILE + 1), (0, 4111 * TILE - 5),
                                     (1, 16385 * TILE), (0, 32768 * TILE), (0, MOST)])
@pytest.mark.parametrize("short", [False, True])
def test_plain(world, begin, n, short):
    ctx, scene, h, cmds, cnt = world
    v = H.view(pyr=(1024, 512))
    cap = n // 40 * 2 + 3 if short else n // 4
    guard = 24 * 64
    cmds.fill_u32(0xABABABAB)
    ctx.cull(h, v, A.PASS_PLAIN, cmds, cnt, capacity=cap, begin=begin, n=n)
    ctx.check_kernels()
    out, total = ctx.read_commands(cmds, cnt, capacity=cap)
    exp, ne = orc.cull(scene, H.view_bytes(v), A.PASS_PLAIN, begin=begin, count=n, capacity=cap, threads=16)
    assert total == ne and (total > cap) == short, (total, ne, cap)
    np.testing.assert_array_equal(H.cmds_u32(out), exp)
    written = min(total, cap) * 6
    after = cmds.download(np.uint32, min(written + guard // 4, cmds.nbytes // 4))[written:]
    assert (after == 0xABABABAB).all()
