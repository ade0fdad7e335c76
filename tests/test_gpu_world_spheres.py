"""Culls read the objects' world-space spheres, which transform updates keep current: after any update, the result
equals the oracle's on the updated transforms."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz
from oracle import pyoracle as orc

from . import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 257, 70001])
@pytest.mark.parametrize("mapping", ["identity", "spare", "pairs", "skewed"])
@pytest.mark.parametrize("surfaces", [16, 65537])
def test_update_reaches_every_object(n, mapping, surfaces):
    """identity: object i uses transform i; spare: the same, with transforms that no object uses (updated too); pairs:
    random transforms, two objects each on average; skewed: one transform for nearly all objects. 65 537 surfaces: the
    32-bit surface ids."""
    sc = bz.synth_scene(31 + n, n, surfaces, 1)
    rng = np.random.default_rng([n, len(mapping)])
    objects, xfs = sc.objects.copy(), sc.transforms.copy()
    if mapping == "spare":
        xfs = np.concatenate([xfs, xfs[:5 if n >= 5 else 1]])
    elif mapping == "pairs":
        objects["transformId"] = rng.integers(0, max(1, n // 2), n, dtype=np.uint32)
    elif mapping == "skewed":
        objects["transformId"] = np.where(np.arange(n) % 1000 == 999, np.arange(n), n - 1).astype(np.uint32)
    v = H.view()
    with bz.Context(0) as ctx:
        h = ctx.scene_create(objects, xfs, sc.surfaces, sc.lods)
        cmds, cnt = ctx.alloc(n * 24), ctx.alloc(4)
        for rounds in range(2):
            ids = np.unique(np.append(rng.integers(0, len(xfs), max(1, n // 3), dtype=np.uint32),
                                      np.uint32(len(xfs) - 1)))
            new = xfs[ids].copy()
            new["pos"] = rng.uniform(-100, 100, (len(ids), 3)).astype(np.float32)
            new["orientation"] = rng.uniform(-1, 1, (len(ids), 4)).astype(np.float32)
            new["scale"] = rng.uniform(0.5, 20, len(ids)).astype(np.float32)
            xfs[ids] = new
            ctx.update_transforms(h, ids, new)
            ctx.cull(h, v, A.PASS_PLAIN, cmds, cnt)
            got, k = ctx.read_commands(cmds, cnt)
            ctx.check_kernels()
            want, kw = orc.cull((objects, xfs, sc.surfaces, sc.lods), H.view_bytes(v), A.PASS_PLAIN)
            assert k == kw
            assert np.array_equal(H.cmds_u32(got), want)


@pytest.mark.parametrize("n", [16383, 16384, 16385, 40000])
@pytest.mark.parametrize("order", ["ascending", "descending", "last twice"])
def test_update_sizes(n, order):
    """One launch for up to 16 384 ascending updates, two for more and for any other order."""
    total = 50000
    sc = bz.synth_scene(97, total, 16, 4)
    rng = np.random.default_rng(n)
    xfs, v = sc.transforms.copy(), H.view()
    ids = np.sort(rng.permutation(total)[:n]).astype(np.uint32)
    if order == "descending":
        ids = np.ascontiguousarray(ids[::-1])
    elif order == "last twice":
        ids[-1] = ids[-2]
    new = xfs[ids].copy()
    new["pos"] = rng.uniform(-100, 100, (n, 3)).astype(np.float32)
    for k, i in enumerate(ids):
        xfs[i] = new[k]
    with bz.Context(0) as ctx:
        h = ctx.scene_create(sc.objects, sc.transforms, sc.surfaces, sc.lods)
        cmds, cnt = ctx.alloc(total * 24), ctx.alloc(4)
        ctx.update_transforms(h, ids, new)
        ctx.cull(h, v, A.PASS_PLAIN, cmds, cnt)
        got, k = ctx.read_commands(cmds, cnt)
        ctx.check_kernels()
        want, kw = orc.cull((sc.objects, xfs, sc.surfaces, sc.lods), H.view_bytes(v), A.PASS_PLAIN)
        assert k == kw and np.array_equal(H.cmds_u32(got), want)
