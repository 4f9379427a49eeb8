"""A launch group that is refused runs as halves, down to single flushes.  A
frame of two flushes whose bins outweigh what a group counts beforehand is
refused under bounds between what its flushes need one by one and what
they need together; it must come out the same there, eagerly and as a captured
frame that loads its target.  A group with a draw that cannot be drawn ends as
flush by flush: what comes before the draw's flush is in the target."""
import numpy as np
import pytest

import rivehip
from streams import BEVEL, StreamBuilder, gradient_limit_stream, rect

pytestmark = pytest.mark.gpu


def wide_strokes(draws=3000, side=1024, segments=140):
    """Zigzags a third of the canvas wide, each with a complex gradient of its
    own: past 2048 of them a second flush starts.  (A translucent rectangle under
    them shows at the right edge how often the frame was drawn.)"""
    rng = np.random.default_rng(3)
    b = StreamBuilder(side, side, clear_color=0xff202020)
    b.draw(b.path(rect(0, 0, side, side)), color=0x40ffffff)
    paths = []
    for _ in range(40):
        pts = rng.uniform(0, [side * .6, side], (segments + 1, 2))
        paths.append(b.path([(0, *map(float, pts[0]))] + [(1, *map(float, p)) for p in pts[1:]]))
    for k in range(draws):
        stops = [(0.0, 0x08000000 | k), (0.5, 0x08ff0000), (1.0, 0x080000ff ^ k << 8)]
        b.draw(paths[k % 40], stroke=side * .3, join=BEVEL, gradient=("linear", 1.0, 1.0, side, side, stops))
    return b


def state(ctx, t, side):
    return (ctx.read_pixels(t, side, side), ctx.last_flush_stats().as_dict(), [ctx.readback(k) for k in range(5)])


def equal(a, b):
    return np.array_equal(a[0], b[0]) and a[1] == b[1] and all(np.array_equal(x, y) for x, y in zip(a[2], b[2]))


@pytest.fixture(scope="module")
def frame_of_two():
    b = wide_strokes()
    s = b.build()
    side = b.width
    ctx = rivehip.Context(0)
    t = ctx.target(side, side)
    assert ctx.render_stream(s, t) == 2
    frame = ctx.last_frame()
    ctx.set_scratch_limit(1)
    ctx.set_scratch_limit(0)
    stats = ctx.reflush_frame(frame, t)
    single = ctx.scratch_bytes()
    ctx.set_scratch_limit(1)
    ctx.set_scratch_limit(0)
    ctx.flush_frame(frame, t)
    ref = state(ctx, t, side)
    joined = ctx.scratch_bytes()
    # what a group of both counts: 108 B a texel and 12 B a cell, a quarter on top
    tiles = (side // 16) ** 2
    counts = sum(-(-st.tess_vertex_count // 2048) * 2048 * 108 + (st.path_count + 1) * tiles * 12 for st in stats) * 5 // 4
    print(f"[fallback] joined {joined} single {single} counted {counts}", flush=True)
    yield ctx, t, side, frame, ref, joined, single, counts
    ctx.set_scratch_limit(0)
    ctx.free_target(t)
    ctx.close()
    del b


@pytest.mark.parametrize("part", [12, 32, 63])
def test_refused_group(frame_of_two, part):
    ctx, t, side, frame, ref, joined, single, counts = frame_of_two
    limit = single + (joined - single) * part // 64
    print(f"[fallback] limit {limit}", flush=True)
    assert counts <= limit // 2 and limit < joined  # so both flushes are tried together, and refused
    ctx.set_scratch_limit(1)
    ctx.set_scratch_limit(limit)
    for _ in range(3):
        ctx.flush_frame(frame, t)
        assert ctx.scratch_bytes() <= limit
        assert equal(ref, state(ctx, t, side))
    ctx.set_scratch_limit(0)


def test_refused_group_of_a_captured_frame(frame_of_two):
    ctx, t, side, frame, ref, joined, single, counts = frame_of_two
    limit = (single + joined) // 2
    print("[fallback] graph", flush=True)
    load = [rivehip.FlushDesc.from_buffer_copy(d) for d in frame]
    load[0].load_action = 1
    ctx.set_scratch_limit(0)
    ctx.flush_frame(frame, t)
    runs = []
    for _ in range(3):
        ctx.flush_frame(load, t)
        runs.append(ctx.read_pixels(t, side, side))
    assert not np.array_equal(runs[0], runs[1])
    ctx.flush_frame(frame, t)
    ctx.set_scratch_limit(1)
    ctx.set_scratch_limit(limit)
    g = ctx.frame_graph(load, t)
    try:
        assert np.array_equal(runs[0], ctx.read_pixels(t, side, side))  # drawn once
        ctx.frame_graph_launch(g)
        assert np.array_equal(runs[1], ctx.read_pixels(t, side, side))
        ctx.set_scratch_limit(0)
        ctx.flush_frame(frame, t)
        ctx.flush_frame(load, t)
        ctx.frame_graph_launch(g)
        assert np.array_equal(runs[1], ctx.read_pixels(t, side, side))
    finally:
        ctx.frame_graph_destroy(g)
    ctx.flush_frame(frame, t)
    assert equal(ref, state(ctx, t, side))


def test_a_draw_that_cannot_be_drawn():
    b = gradient_limit_stream(2200)
    s = b.build()
    w, h = b.width, b.height
    print("[fallback] bad draw", flush=True)
    ctx = rivehip.Context(0)
    t = ctx.target(w, h)
    try:
        assert ctx.render_stream(s, t) == 2
        frame = ctx.last_frame()
        ctx.flush_frame(frame[:1], t)
        first = ctx.read_pixels(t, w, h)
        draws = np.concatenate([ctx.readback(3).view(rivehip.DRAW)])
        ctx.flush(frame[1])
        draws = np.concatenate([draws, ctx.readback(3).view(rivehip.DRAW)])
        both = ctx.read_pixels(t, w, h)
        assert not np.array_equal(first, both)
        bad = draws.copy()
        bad[-1]["image_index"] = 3  # the frame has no images
        ctx.upload("draw", bad)
        with pytest.raises(RuntimeError) as e:
            ctx.flush_frame(frame, t)
        assert "out of range" in str(e.value)
        assert np.array_equal(first, ctx.read_pixels(t, w, h))
        ctx.upload("draw", draws)
        ctx.flush_frame(frame, t)
        assert np.array_equal(both, ctx.read_pixels(t, w, h))
    finally:
        ctx.free_target(t)
        ctx.close()
