"""Pyramid builds whose depth image holds more than two texels per base texel (each footprint's row is one load, a texel
early at the row's end), depth images one to three texels wide, and builds of a single level, of few levels and of a
last level around the size where a build by regions ends; bit-exact against the oracle. Needs a GPU."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import cull as bz
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu

# depth w, h, base w, h, mips
SHAPES = [(1, 9, 4, 4, 3), (2, 2, 8, 8, 4), (3, 3, 16, 1, 5), (5, 4, 2, 2, 2), (65, 64, 32, 32, 6), (97, 33, 32, 32, 1),
          (515, 300, 128, 64, 8), (1000, 999, 256, 256, 9), (937, 41, 128, 32, 2), (4096, 1024, 1024, 256, 11),
          (300, 2000, 64, 512, 10), (2048, 512, 1024, 256, 1), (640, 360, 512, 256, 1), (240, 136, 120, 68, 1),
          (240, 136, 120, 68, 2), (33, 17, 7, 5, 1), (1600, 1280, 800, 640, 4), (1602, 1280, 801, 640, 4),
          (1920, 1080, 960, 540, 4), (1920, 1080, 960, 540, 10)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("offset", [0, 4])
def test_ratios(shape, offset):
    w, h, bw, bh, mips = shape
    rng = np.random.default_rng(w * h + mips)
    depth = rng.uniform(0.0, 1.0, (h, w)).astype(np.float32)
    depth[rng.random((h, w)) < 0.02] = np.inf
    with bz.Context(0) as ctx:
        buf = ctx.alloc(depth.nbytes + offset)  # the image ends where the allocation does
        buf.upload(np.concatenate([np.zeros(offset // 4, np.float32), depth.reshape(-1)]))
        p = ctx.pyramid_create(bw, bh, mips)
        want = orc.pyramid_build(depth, bw, bh, mips).view(np.uint32)
        for _ in range(2):
            ctx.pyramid_build(p, buf.ptr + offset, w, h)
            ctx.check_kernels()
            got, _ = ctx.pyramid_read(p, mips)
            np.testing.assert_array_equal(got.view(np.uint32), want)
        ctx.pyramid_build_batch([(p, buf.ptr + offset, w, h)])
        ctx.check_kernels()
        got, _ = ctx.pyramid_read(p, mips)
        np.testing.assert_array_equal(got.view(np.uint32), want)
