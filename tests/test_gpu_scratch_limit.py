"""A context's device scratch has a bound that the caller sets.  A frame of two
flushes must come out the same, with the same statistics and intermediates, in
one launch group and in the several that a lower bound leaves; what is held
stays within the bound; and a flush that cannot fit is refused, after which the
context works on."""
import numpy as np
import pytest

import rivehip
from streams import MITER, StreamBuilder

pytestmark = pytest.mark.gpu


def wide_strokes(draws=3000, w=400, h=300, segments=12):
    """Long wide zigzags, each with a complex gradient of its own: past 2048 of
    them a second flush starts.  Their bins outweigh their tessellation."""
    rng = np.random.default_rng(3)
    b = StreamBuilder(w, h, clear_color=0xff202020)
    paths = []
    for _ in range(40):
        pts = rng.uniform(0, [w, h], (segments + 1, 2))
        paths.append(b.path([(0, *map(float, pts[0]))] + [(1, *map(float, p)) for p in pts[1:]]))
    for k in range(draws):
        stops = [(0.0, 0x20000000 | k), (0.5, 0x20ff0000), (1.0, 0x200000ff ^ k << 8)]
        b.draw(paths[k % 40], stroke=60.0, join=MITER, gradient=("linear", 1.0, 1.0, float(w), float(h), stops))
    return b


def state(ctx, t, w, h):
    return (ctx.read_pixels(t, w, h), ctx.last_flush_stats().as_dict(), [ctx.readback(k) for k in range(5)])


def equal(a, b):
    return np.array_equal(a[0], b[0]) and a[1] == b[1] and all(np.array_equal(x, y) for x, y in zip(a[2], b[2]))


@pytest.fixture(scope="module")
def two_flushes():
    """A frame of two flushes in a context of its own, what it draws and holds
    in one group, and what a context holds that draws it flush by flush."""
    b = wide_strokes()
    s = b.build()
    w, h = b.width, b.height
    ctx = rivehip.Context(0)
    t = ctx.target(w, h)
    assert ctx.render_stream(s, t) == 2
    frame = ctx.last_frame()
    ctx.flush_frame(frame, t)
    ref = state(ctx, t, w, h)
    joined = ctx.scratch_bytes()
    ctx.set_scratch_limit(1 << 40)
    assert ctx.scratch_bytes() == joined  # a bound above what is held changes nothing
    ctx.set_scratch_limit(1)
    assert ctx.scratch_bytes() == 0
    ctx.set_scratch_limit(0)
    ctx.reflush_frame(frame, t)
    assert equal(ref, state(ctx, t, w, h))
    single = ctx.scratch_bytes()
    print(f"[scratch] joined {joined} single {single}", flush=True)
    yield ctx, t, w, h, frame, ref, joined, single
    ctx.set_scratch_limit(0)
    ctx.free_target(t)
    ctx.close()
    del b


def test_a_lower_bound_runs_in_several_groups(two_flushes):
    ctx, t, w, h, frame, ref, joined, single = two_flushes
    limit = single + single // 8
    print(f"[scratch] limit {limit}", flush=True)
    assert limit < joined
    ctx.set_scratch_limit(1)
    ctx.set_scratch_limit(limit)
    for _ in range(2):
        ctx.flush_frame(frame, t)
        assert equal(ref, state(ctx, t, w, h))
        assert ctx.scratch_bytes() <= limit
    ctx.set_scratch_limit(0)


def test_a_flush_beyond_the_bound_is_refused(two_flushes):
    ctx, t, w, h, frame, ref, joined, single = two_flushes
    ctx.set_scratch_limit(single // 4)
    print("[scratch] refused", flush=True)
    with pytest.raises(RuntimeError) as e:
        ctx.flush_frame(frame, t)
    assert "scratch limit" in str(e.value)
    assert ctx.scratch_bytes() <= single // 4
    ctx.set_scratch_limit(0)
    ctx.flush_frame(frame, t)
    assert equal(ref, state(ctx, t, w, h))
