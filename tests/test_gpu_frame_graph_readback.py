"""A captured frame keeps its intermediates in its own buffers, so after a
capture there are none of a last flush to read back: every readback is empty
(a frame of one flush, and one whose last flush lay behind others in its
buffers).  An eager frame afterwards has its intermediates again."""
import numpy as np
import pytest

import rivehip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("draws", [40, 2600])
def test_nothing_to_read_back_after_a_capture(draws):
    print(f"[graph-readback] {draws}", flush=True)
    w, h = 640, 400
    s = rivehip.generate_stream(2, seed=5, width=w, height=h, draw_count=draws)
    ctx = rivehip.Context(0)
    t = ctx.target(w, h)
    g = None
    try:
        ctx.render_stream(s, t)
        frame = ctx.last_frame()
        ctx.flush_frame(frame, t)
        eager = ctx.read_pixels(t, w, h)
        before = [ctx.readback(k) for k in range(6)]
        assert all(b.size for b in before)
        g = ctx.frame_graph(frame, t)
        assert [ctx.readback(k).size for k in range(6)] == [0] * 6
        ctx.frame_graph_launch(g)
        assert np.array_equal(eager, ctx.read_pixels(t, w, h))
        ctx.flush_frame(frame, t)
        for k, a in enumerate(before):
            assert np.array_equal(a, ctx.readback(k)), f"readback {k}"
    finally:
        if g is not None:
            ctx.frame_graph_destroy(g)
        ctx.free_target(t)
        ctx.close()
        rivehip.free_stream(s)
