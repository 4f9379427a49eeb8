"""The raster's two row forms: int32 for primitives near their tile (vertices
within 64 px; feathered segments within 128 px with edges up to 101 px) and
double for the rest.  Polygons and strokes whose straight edges lie on either
side of those limits, at offsets on and off tile corners, and feathers of
radii around them must match the oracle within 2/255 on all but 0.1% of pixels and
8/255 everywhere, as the scenes of test_gpu_random_scenes.py do.  (Feathers whose radius exceeds the shape are left out: there the
oracle's quarter-resolution atlas and a direct evaluation differ by design.)"""
import numpy as np
import pytest

import oracle_binding as ob
import rivehip
from streams import CLOCKWISE, MITER, StreamBuilder

pytestmark = pytest.mark.gpu


def zigzag(length, x, y, n, closed):
    """n edges of `length` px turning back and forth, slowly drifting."""
    pts = [(x, y)]
    for k in range(n):
        a = (0.07 + 0.31 * k) if k % 2 == 0 else np.pi + 0.31 * k - 0.2
        x, y = x + length * np.cos(a), y + length * np.sin(a)
        pts.append((float(x), float(y)))
    return [(0, *pts[0])] + [(1, *p) for p in pts[1:]] + ([(5,)] if closed else [])


def compare(ctx, b):
    s = b.build()
    f = ob.OracleFlush(s)
    t = ctx.target(b.width, b.height)
    try:
        ref, _ = f.render()
        ctx.render_stream(s, t)
        out = ctx.read_pixels(t, b.width, b.height)
    finally:
        ctx.free_target(t)
        f.close()
    d = np.abs(out.astype(np.int32) - ref.astype(np.int32)).max(axis=2)
    assert out.any()
    assert d.max() <= 8 and (d > 2).mean() <= 1e-3, f"max {d.max()}, frac>2 {(d > 2).mean()}"


@pytest.mark.parametrize("length", [15.99, 16.0, 47.5, 63.9, 64.0, 64.3, 100.0, 240.0, 5000.0])
def test_edges_around_the_near_limit(hip_ctx, length):
    print(f"[rows] {length}", flush=True)
    b = StreamBuilder(210, 190, clear_color=0xff101010)
    for k, (x, y) in enumerate([(96.0, 80.0), (100.37, 91.7), (16.0, 15.996), (180.2, 170.9)]):
        b.draw(b.path(zigzag(length, x, y, 7, True), k % 2), color=0xa0ff8040 + 0x30507 * k)
        b.draw(b.path(zigzag(length, x + 5, y - 3, 5, False)), color=0xc040a0ff - 0x30507 * k, stroke=[1., 6., 40., .4][k],
               join=MITER)
    compare(hip_ctx, b)


@pytest.mark.parametrize("feather", [2.0, 20.0, 41.0, 60.0, 84.0])
def test_feathers_around_the_near_limit(hip_ctx, feather):
    print(f"[rows] feather {feather}", flush=True)
    b = StreamBuilder(230, 210, clear_color=0xff101010)
    b.draw(b.path([(0, 60, 50), (1, 170, 64), (4, 200, 130, 120, 190, 70, 150), (5,)], CLOCKWISE), color=0xffe0a030,
           feather=feather)
    b.draw(b.path(zigzag(90.0, 40.0, 100.0, 3, False)), color=0xc040a0ff, stroke=9.0, feather=feather / 4)
    compare(hip_ctx, b)
