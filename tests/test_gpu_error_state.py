"""A HIP call that fails is reported once, by the call that made it: what runs
after it on the context must not see its error.  An allocation far beyond the
card is refused by the runtime without touching it; the frames, images and
targets after that must come out as before."""
import numpy as np
import pytest

import rivehip

pytestmark = pytest.mark.gpu


def test_refused_allocation_is_reported_once(hip_ctx):
    print("[error-state] refused allocation", flush=True)
    s = rivehip.generate_stream(1, draw_count=30, width=128, height=96)
    t = hip_ctx.target(128, 96)
    rgba = np.full((33, 35, 4), 200, np.uint8)
    try:
        hip_ctx.render_stream(s, t)
        before = hip_ctx.read_pixels(t, 128, 96)
        span = rivehip.BUFFER["tess_span"]  # not read by GEOMETRY flushes
        with pytest.raises(RuntimeError):
            rivehip.check(hip_ctx.L.rive_hip_buffer_resize(hip_ctx.h, span, 1 << 50))
        hip_ctx.render_stream(s, t)
        assert np.array_equal(before, hip_ctx.read_pixels(t, 128, 96))
        with pytest.raises(RuntimeError):
            rivehip.check(hip_ctx.L.rive_hip_buffer_resize(hip_ctx.h, span, 1 << 50))
        im = hip_ctx.image(rgba)
        assert (hip_ctx.image_read(im, 2) == 200).all()
        hip_ctx.free_image(im)
        hip_ctx.upload("tess_span", np.zeros(16, np.uint8))
    finally:
        hip_ctx.free_target(t)
        rivehip.free_stream(s)
