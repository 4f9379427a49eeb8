"""Binning puts the segments that span tile rows and columns, or cross a tile
line, aside and takes them 64 a wave at a time, in workgroups whose size follows
the number of draws and the canvas.  Contours of long diagonals (every segment
put aside), of short segments (few) and of both, in counts around a wave's queue
and on either side of each workgroup size, against the oracle: within 2/255 on
all but 0.1% of pixels and 8/255 everywhere.

Parity unpinned: a thousand long diagonals in one path, and feathered stars of
more than 65.  Every edge adds what its vertices' snapping to 1/256 px moves its
border, so the sum of so many a pixel leaves that tolerance whatever bins them.
The diagonals are binned both ways instead -- in LDS, and by global atomics as a
path with guard-box pieces is -- and must give the same bytes."""
import numpy as np
import pytest

import oracle_binding as ob
from streams import EVENODD, NONZERO, StreamBuilder

pytestmark = pytest.mark.gpu


def check(ctx, b):
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
    assert d.max() <= 8 and (d > 2).mean() <= 1e-3, f"max {d.max()}, frac>2 {(d > 2).mean()}"


# (1100 long ones: test_routes_agree)
COUNTS = [(k, n) for k in ("long", "short", "mixed") for n in (3, 63, 64, 65, 112, 113, 400, 1100)
          if (k, n) != ("long", 1100)]


@pytest.mark.parametrize("feather", [0.0, 30.0])
@pytest.mark.parametrize("kind,n", COUNTS)
def test_segments_put_aside(hip_ctx, kind, n, feather):
    print(f"[bin-walk] {kind} {n} {feather}", flush=True)
    rng = np.random.default_rng(n)
    w, h = 333, 271
    b = StreamBuilder(w, h, clear_color=0xff203040)
    x, y = w / 2, h / 2
    cmds = [(0, x, y)]
    for k in range(n):
        if kind == "long" or (kind == "mixed" and rng.random() < .3):
            x, y = float(rng.uniform(-20, w + 20)), float(rng.uniform(-20, h + 20))
        else:
            x, y = x + float(rng.uniform(-7, 7)), y + float(rng.uniform(-7, 7))
        cmds.append((1, x, y))
    # (feathered stars of more segments: parity unpinned)
    b.draw(b.path(cmds[:1 + (n if feather == 0 else min(n, 65))] + [(5,)], fill_rule=EVENODD if n % 2 else NONZERO),
           color=0xc0f08020, feather=feather)
    check(hip_ctx, b)


@pytest.mark.parametrize("n", [1100, 4001])
def test_routes_agree(hip_ctx, n):
    """A spike right of the canvas, out of the guard box and back, gives the path
    pieces, so that it is binned by global atomics; on the canvas nothing changes."""
    print(f"[bin-walk] routes {n}", flush=True)
    rng = np.random.default_rng(n)
    w, h = 333, 271
    pts = rng.uniform([-20, -20], [w + 20, h + 20], (n, 2))
    head = [(0, w / 2, h / 2)] + [(1, float(x), float(y)) for x, y in pts] + [(1, w + 140., h / 2), (1, w + 160., h / 2 + 10)]
    out = []
    for spike in ([], [(1, 60000., h / 2 + 10), (1, w + 160., h / 2 + 10)]):
        b = StreamBuilder(w, h, clear_color=0xff203040)
        b.draw(b.path(head + spike + [(1, w + 180., h / 2), (5,)], fill_rule=EVENODD if n % 2 else NONZERO),
               color=0xc0f08020)
        t = hip_ctx.target(w, h)
        try:
            hip_ctx.render_stream(b.build(), t)
            assert (hip_ctx.last_flush_stats().guard_pieces > 0) == bool(spike)
            out.append(hip_ctx.read_pixels(t, w, h))
        finally:
            hip_ctx.free_target(t)
    assert len(np.unique(out[0].reshape(-1, 4), axis=0)) > 100
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("w,h,n", [(160, 128, 512), (160, 128, 513), (160, 128, 2048), (160, 128, 2049),
                                   (1040, 1024, 513)])
def test_workgroup_sizes(hip_ctx, w, h, n):
    print(f"[bin-walk] {w}x{h} {n} draws", flush=True)
    rng = np.random.default_rng(n)
    b = StreamBuilder(w, h, clear_color=0xff203040)
    for k in range(n):
        x, y = rng.uniform(0, [w, h])
        r = rng.uniform(2, 40, 3)
        a = rng.uniform(0, 6.28) + np.array([0, 2.1, 4.2])
        pts = [(1, float(x + r[q] * np.cos(a[q])), float(y + r[q] * np.sin(a[q]))) for q in range(3)]
        b.draw(b.path([(0, *pts[0][1:]), *pts[1:], (5,)]), color=int(rng.integers(0, 1 << 24)) | 0xa0000000)
    check(hip_ctx, b)
