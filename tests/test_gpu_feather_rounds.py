"""A batch of feathered segments with more rows than the raster's owner table
holds is taken in rounds, and the feather is sampled from a table of texel pairs
in LDS.  Small tight contours whose every segment spans all rows of a tile, with
and without join ends (corners and smooth curves), as fills and strokes, against
the oracle: within 2/255 on all but 0.1% of pixels and 8/255 everywhere."""
import numpy as np
import pytest

import oracle_binding as ob
from streams import ROUND, ROUND_CAP, StreamBuilder

pytestmark = pytest.mark.gpu


def star(n, cx, cy, r0, r1):
    a = np.arange(n) * (2 * np.pi / n)
    r = np.where(np.arange(n) % 2, r0, r1)
    return [(0 if k == 0 else 1, float(cx + r[k] * np.cos(a[k])), float(cy + r[k] * np.sin(a[k]))) for k in range(n)]


def flower(n, cx, cy, r0, r1):
    a = np.arange(3 * n + 1) * (2 * np.pi / (3 * n))
    r = r0 + (r1 - r0) * (.5 + .5 * np.cos(n * a))
    pts = [(float(cx + r[k] * np.cos(a[k])), float(cy + r[k] * np.sin(a[k]))) for k in range(3 * n + 1)]
    return [(0, *pts[0])] + [(4, *pts[3 * k + 1], *pts[3 * k + 2], *pts[3 * k + 3]) for k in range(n)]


@pytest.mark.parametrize("feather", [6.0, 24.0])
@pytest.mark.parametrize("kind,n", [("star", 20), ("star", 130), ("star", 500), ("flower", 60), ("stroke", 130)])
def test_rounds(hip_ctx, kind, n, feather):
    w, h = 53, 39
    b = StreamBuilder(w, h, clear_color=0xff303030)
    for k in range(2):
        make = flower if kind == "flower" else star
        p = b.path(make(n, 24 + 5 * k, 19, 5.0 + k, 9.0 + 2 * k) + [(5,)])
        kw = dict(stroke=3.0, join=ROUND, cap=ROUND_CAP) if kind == "stroke" else {}
        b.draw(p, color=(0xd0e04020, 0x8020c0f0)[k], feather=feather, **kw)
    s = b.build()
    print(f"[feather-rounds] {kind} {n} {feather}", flush=True)
    f = ob.OracleFlush(s)
    t = hip_ctx.target(w, h)
    try:
        ref, _ = f.render()
        hip_ctx.render_stream(s, t)
        out = hip_ctx.read_pixels(t, w, h)
    finally:
        hip_ctx.free_target(t)
        f.close()
    d = np.abs(out.astype(np.int32) - ref.astype(np.int32)).max(axis=2)
    assert d.max() <= 8 and (d > 2).mean() <= 1e-3, f"max {d.max()}, frac>2 {(d > 2).mean()}"
