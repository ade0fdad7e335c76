"""Min-depth pyramids at the edges of their tiles: every shape, one and many at a time, bit-exact against the oracle,
with infinities, NaN and both zeros among the depths.

With NaN a minimum depends on the order of its operands (`y < x ? y : x` keeps x when either is NaN). The kernels take
the minimum of the two rows' minima, the oracle one texel after another; images with NaN are compared with the kernels'
order, restated in numpy."""
from __future__ import annotations

import numpy as np
import pytest

from blitzen_amd import cull as bz
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu

# (depth w, h, base w, h, mips): single texels and rows, extents below, at and just over a 32-texel tile, tile images of
# one row, of one column, with an empty tail and with the largest one; exact 2:1 and general ratios; more mips than the
# extent halves
SHAPES = [(1, 1, 1, 1, 1), (2, 2, 1, 1, 3), (5, 3, 2, 1, 4), (3, 130, 1, 64, 9), (130, 3, 64, 1, 7), (31, 33, 16, 16, 5),
          (64, 64, 32, 32, 6), (64, 64, 32, 32, 9), (70, 50, 64, 32, 7), (128, 64, 64, 32, 5), (100, 200, 32, 128, 8),
          (512, 4, 256, 2, 9), (700, 1, 512, 1, 10), (256, 256, 128, 128, 3), (1366, 768, 1024, 512, 11),
          (4096, 4096, 2048, 2048, 12), (3001, 1500, 2048, 1024, 12)]
# not powers of two: regions of one tile and of many, odd halves, one texel wide or high, fewer and more levels than the
# regions hold, the largest image of the last level (120 x 67) and one that takes a launch per level (128 x 68)
SHAPES += [(5, 5, 3, 5, 3), (37, 23, 18, 11, 5), (101, 7, 99, 1, 7), (7, 3000, 1, 1500, 11), (1000, 777, 500, 388, 9),
           (640, 360, 321, 179, 1), (640, 360, 320, 181, 4), (1600, 900, 800, 450, 10), (1366, 768, 683, 384, 12),
           (3840, 2160, 1920, 1080, 11), (4100, 2200, 2050, 1100, 12)]


def image(w, h, seed, odd_values):
    rng = np.random.default_rng(seed)
    d = rng.uniform(0.0, 1.0, (h, w)).astype(np.float32)
    if odd_values:
        pick = rng.random((h, w))
        for k, x in enumerate((np.inf, -np.inf, np.nan, 0.0, -0.0)):
            d[(pick > 0.1 * k) & (pick < 0.1 * k + 0.08)] = x
    return d


def axis(n_dst, n_src):
    """Texels of non-zero weight per destination texel, from float32 sample positions."""
    f = np.float32
    t = (np.arange(n_dst).astype(f) + f(0.5)) / f(n_dst) * f(n_src) - f(0.5)
    lo = np.floor(t)
    i0 = np.clip(lo, 0, n_src - 1).astype(int)
    return i0, np.where(t - lo > 0, np.clip(lo + 1, 0, n_src - 1).astype(int), i0)


def first_min(x, y):
    return np.where(y < x, y, x)


def by_rows(depth, bw, bh, mips):
    src, out = depth, []
    for k in range(mips):
        (x0, x1), (y0, y1) = axis(max(1, bw >> k), src.shape[1]), axis(max(1, bh >> k), src.shape[0])
        top, bottom = src[y0], src[y1]
        src = first_min(first_min(top[:, x0], top[:, x1]), first_min(bottom[:, x0], bottom[:, x1]))
        out.append(src.reshape(-1))
    return np.concatenate(out)


def expected(depth, bw, bh, mips):
    want = by_rows(depth, bw, bh, mips).view(np.uint32)
    if not np.isnan(depth).any():
        assert np.array_equal(want, orc.pyramid_build(depth, bw, bh, mips).view(np.uint32))
    return want


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("odd_values", [False, True])
@pytest.mark.parametrize("offset", [0, 4, 8])
def test_one_pyramid(shape, odd_values, offset):
    """offset: bytes from the allocation's start to the depth image (its alignment chooses the loads)."""
    w, h, bw, bh, mips = shape
    if offset and w * h > 1 << 20:
        pytest.skip("alignment is covered by the smaller shapes")
    depth = image(w, h, w * h + mips, odd_values)
    with bz.Context(0) as ctx:
        buf = ctx.alloc(depth.nbytes + 16)
        buf.upload(np.concatenate([np.zeros(offset // 4, np.float32), depth.reshape(-1)]))
        p = ctx.pyramid_create(bw, bh, mips)
        for _ in range(2):  # the second build starts from the hand-off words the first one left
            ctx.pyramid_build(p, buf.ptr + offset, w, h)
            ctx.check_kernels()
            got, _ = ctx.pyramid_read(p, mips)
            assert np.array_equal(got.view(np.uint32), expected(depth, bw, bh, mips))


def test_all_shapes_in_one_batch():
    with bz.Context(0) as ctx:
        jobs, want = [], []
        for k, (w, h, bw, bh, mips) in enumerate(SHAPES):
            depth = image(w, h, 77 + k, bool(k & 1))
            buf = ctx.alloc(depth.nbytes)
            buf.upload(depth)
            p = ctx.pyramid_create(bw, bh, mips)
            jobs.append((p, buf.ptr, w, h))
            want.append((p, mips, expected(depth, bw, bh, mips)))
        for _ in range(2):
            ctx.pyramid_build_batch(jobs)
            ctx.check_kernels()
            for p, mips, exp in want:
                got, _ = ctx.pyramid_read(p, mips)
                assert np.array_equal(got.view(np.uint32), exp)
