"""A tuning that a caller sets or loads is taken as it is, also one of the values that the built-in choice by the number of
objects is reported with; that choice is put back by the value that bz_get_tuning gave. Needs a GPU."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz
from oracle import pyoracle as orc
from tests import helpers as H

pytestmark = pytest.mark.gpu


def fields(t):
    return t.block, t.items, t.grid_per_cu, t.reserved


def test_built_in_choice_is_told_from_its_values():
    n = 70000
    sc, v = bz.synth_scene(23, n, 64, 4), H.view()
    want, k = orc.cull(H.as_tuple(sc), H.view_bytes(v), A.PASS_PLAIN, threads=8)
    with bz.Context(0) as ctx:
        h = ctx.scene_create(*H.as_tuple(sc))
        cmds, cnt = ctx.alloc(n * 24), ctx.alloc(4)
        built_in = ctx.get_tuning(0)
        assert fields(built_in) == (512, 2, 0, A.TUNING_BY_SIZE)
        for t in ((512, 2, 0, 0), (512, 2, 1, 0), fields(built_in)):
            ctx.set_tuning(0, *t)
            assert fields(ctx.get_tuning(0)) == t
            ctx.cull(h, v, A.PASS_PLAIN, cmds, cnt)
            got, total = ctx.read_commands(cmds, cnt)
            assert total == k
            np.testing.assert_array_equal(H.cmds_u32(got), want)


@pytest.mark.parametrize("entry,want", [("", (512, 2, 0, 0)), (', "by_size": 1', (512, 2, 0, A.TUNING_BY_SIZE))])
def test_loaded_tunings(tmp_path, entry, want):
    """A file's entry is in force as it stands; a choice timed here is read back as it was."""
    n = 40000
    sc, v = bz.synth_scene(24, n, 64, 4), H.view()
    with bz.Context(0) as ctx:
        h = ctx.scene_create(*H.as_tuple(sc))
        cmds, cnt = ctx.alloc(n * 24), ctx.alloc(4)
        job = ctx.view_job(h, v, A.PASS_PLAIN, cmds, cnt)
        cache = tmp_path / "tune.json"
        first = ctx.autotune(0, [job], cache_path=str(cache))
        assert fields(ctx.get_tuning(0)) == fields(first)
        line = next(x for x in cache.read_text().splitlines() if "|k0|" in x)
        ctx.set_tuning(0, 256, 4)
        assert fields(ctx.autotune(0, [job], cache_path=str(cache))) == fields(first)
        name = line.split('"')[1]
        cache.write_text(f'{{\n  "{name}": {{"block": 512, "items": 2, "grid_per_cu": 0, "us": 9.500{entry}}}\n}}\n')
        assert fields(ctx.autotune(0, [job], cache_path=str(cache))) == want
        assert fields(ctx.get_tuning(0)) == want
