"""Updates of transforms that many objects use: lists of objects around the lengths at which a workgroup takes fewer updates,
at which a list is cut into pieces (64, 256, 1024 objects) and at the pieces' ends (256), in one launch and in two; every
object's sphere follows, bit-exact against the oracle on the updated transforms. Needs a GPU."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz
from oracle import pyoracle as orc
from tests import helpers as H

pytestmark = pytest.mark.gpu


def lengths(kind):
    """Objects of each transform."""
    rng = np.random.default_rng(len(kind))
    if kind == "mean 1":  # 256 updates a workgroup, lists up to 64 in one launch
        return np.concatenate([np.ones(30000, int), [0, 63, 64, 65, 255, 256, 257, 512, 513, 0]])
    if kind == "mean 5":  # 64 updates, up to 256
        return np.concatenate([rng.integers(0, 11, 4000), [255, 256, 257, 769, 0]])
    if kind == "mean 20":  # 16 updates, up to 1024
        return np.concatenate([rng.integers(10, 31, 2000), [0, 1023, 1024, 1025]])
    if kind == "mean 200":  # 4 updates, up to 1024
        return np.concatenate([rng.integers(100, 301, 300), [1024, 1025, 5000]])
    return np.array([70001])  # one transform for all


@pytest.mark.parametrize("kind", ["mean 1", "mean 5", "mean 20", "mean 200", "all"])
@pytest.mark.parametrize("order", ["ascending", "shuffled", "repeated"])
def test_every_object_follows(kind, order):
    per = lengths(kind)
    rng = np.random.default_rng([len(kind), len(order)])
    n, nx = int(per.sum()), len(per)
    sc = bz.synth_scene(7, n, 16, 4)
    objects, xfs = sc.objects.copy(), sc.transforms[:nx].copy()
    objects["transformId"] = rng.permutation(np.repeat(np.arange(nx), per)).astype(np.uint32)
    v = H.view()
    with bz.Context(0) as ctx:
        h = ctx.scene_create(objects, xfs, sc.surfaces, sc.lods)
        cmds, cnt = ctx.alloc(n * 24), ctx.alloc(4)
        for part in (1.0, 0.3, 0.0):
            ids = np.flatnonzero(rng.random(nx) < part) if part else np.array([nx - 1])
            ids = np.union1d(ids, [nx - 1]).astype(np.uint32)
            if order == "shuffled":
                rng.shuffle(ids)
            elif order == "repeated":
                ids = np.concatenate([ids, ids[::-1]])
            new = xfs[ids].copy()
            new["pos"] = rng.uniform(-100, 100, (len(ids), 3)).astype(np.float32)
            new["orientation"] = rng.uniform(-1, 1, (len(ids), 4)).astype(np.float32)
            new["scale"] = rng.uniform(0.5, 20, len(ids)).astype(np.float32)
            for k, i in enumerate(ids):  # the last occurrence of an id wins
                xfs[i] = new[k]
            ctx.update_transforms(h, ids, new)
            ctx.cull(h, v, A.PASS_PLAIN, cmds, cnt)
            got, k = ctx.read_commands(cmds, cnt)
            ctx.check_kernels()
            want, kw = orc.cull((objects, xfs, sc.surfaces, sc.lods), H.view_bytes(v), A.PASS_PLAIN, threads=8)
            assert k == kw
            np.testing.assert_array_equal(H.cmds_u32(got), want)
