"""A stream whose only calls so far were small: a pass of up to 2^20 objects can still be captured from it (nothing has to
grow), and its replays equal the oracle. Needs a GPU."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz
from blitzen_amd.hip import StreamGraph
from oracle import pyoracle as orc
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [327681, 1 << 20])
def test_large_pass_captured_after_a_small_one(n):
    sc, v = bz.synth_scene(19, n, 64, 4), H.view()
    with bz.Context(0) as ctx:
        h = ctx.scene_create(*H.as_tuple(sc))
        cmds, cnt, s = ctx.alloc(n * 24), ctx.alloc(4), ctx.stream()
        ctx.cull(h, v, A.PASS_PLAIN, cmds, cnt, capacity=n, begin=0, n=1000, stream=s)
        g = StreamGraph(s, lambda: ctx.cull(h, v, A.PASS_PLAIN, cmds, cnt, capacity=n, stream=s))
        want, k = orc.cull(H.as_tuple(sc), H.view_bytes(v), A.PASS_PLAIN, capacity=n, threads=8)
        for _ in range(2):
            ctx.cull(h, v, A.PASS_PLAIN, cmds, cnt, capacity=n, begin=0, n=1000, stream=s)
            g.launch(s)
            got, total = ctx.read_commands(cmds, cnt, capacity=n, stream=s)
            assert total == k
            np.testing.assert_array_equal(H.cmds_u32(got), want)
        ctx.check_kernels(s)
