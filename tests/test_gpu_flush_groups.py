"""A frame's logical flushes run as one launch of every pass.  The frame must
equal its flushes issued one by one, bit for bit, and leave the last flush's
statistics and intermediates as those do: frames of several flushes with
clips, gradients and strokes, the 2048-gradient-row and 30 719-path splits; a
split frame with images is held to the oracle.  Flushes that cannot be joined (another dither setting)
run on their own."""
import numpy as np
import pytest

import oracle_binding as ob
import rivehip
from streams import gradient_limit_stream, pixel_rects_stream, rect

pytestmark = pytest.mark.gpu


def compare(ctx, stream, w, h, change=None):
    t, one = ctx.target(w, h), ctx.target(w, h)
    try:
        n = ctx.render_stream(stream, t)
        assert n > 1
        frame = ctx.last_frame()
        if change is not None:
            change(frame)
        ctx.flush_frame(frame, t)
        joined = ctx.read_pixels(t, w, h)
        st = ctx.last_flush_stats().as_dict()
        kinds = (0, 1, 2, 3, 4) if st["grad_span_count"] else (0, 1, 2, 3)  # no spans, no ramps
        mid = [ctx.readback(k) for k in kinds]
        stats = ctx.reflush_frame(frame, one)
        assert np.array_equal(joined, ctx.read_pixels(one, w, h))
        assert joined.any()
        assert st == stats[-1].as_dict()
        for k, a, b in zip(kinds, mid, [ctx.readback(k) for k in kinds]):
            assert np.array_equal(a, b), f"readback {k}"
    finally:
        ctx.free_target(t)
        ctx.free_target(one)


@pytest.mark.parametrize("w,h,draws", [(1280, 720, 2600), (333, 517, 5200)])
def test_joined_flushes_equal_single_ones(hip_ctx, w, h, draws):
    print(f"[groups] {w}x{h} {draws}", flush=True)
    s = rivehip.generate_stream(2, seed=17, width=w, height=h, draw_count=draws)
    try:
        compare(hip_ctx, s, w, h)
    finally:
        rivehip.free_stream(s)


def test_images_of_both_flushes(hip_ctx):
    """Images and gradients drawn in each of two flushes, against the oracle."""
    print("[groups] images", flush=True)
    b, _ = pixel_rects_stream(30740)
    rng = np.random.default_rng(5)
    ims = [b.image(np.concatenate([rng.integers(0, 255, (8, 8, 3)), np.full((8, 8, 1), 255)], 2)) for _ in range(3)]
    p = b.path(rect(100, 20, 220, 90))
    stops = [(0.0, 0x80ff0000), (0.5, 0xff00ff00), (1.0, 0x400000ff)]
    tail = b.draws
    b.draws = []
    for k, at in ((0, 10), (1, 70)):
        b.draw_image(ims[k], matrix=(5., 0., 0., 5., float(at), 15.), sampler=9)
    b.draw(p, gradient=("linear", 100., 0., 220., 0., stops))
    b.draws += tail[:-12]
    b.draw_image(ims[2], matrix=(4., 1., -1., 4., 130., 50.), sampler=9, opacity=.7)
    b.draw_image(ims[0], matrix=(2., 0., 0., 2., 30., 60.))
    b.draw(p, gradient=("linear", 0., 20., 0., 90., [(o, c ^ 0xffffff) for o, c in stops]), clips=(p,))
    b.draws += tail[-12:]
    s = b.build()
    f = ob.OracleFlush(s)
    t = hip_ctx.target(b.width, b.height)
    try:
        assert f.flush_count == 2
        ref, _ = f.render()
        assert hip_ctx.render_stream(s, t) == 2
        out = hip_ctx.read_pixels(t, b.width, b.height)
    finally:
        hip_ctx.free_target(t)
        f.close()
    d = np.abs(out.astype(np.int32) - ref.astype(np.int32)).max(axis=2)
    assert d.max() <= 8 and (d > 2).mean() <= 1e-3, f"max {d.max()}, frac>2 {(d > 2).mean()}"


@pytest.mark.parametrize("make", [lambda: gradient_limit_stream(), lambda: pixel_rects_stream(30800)[0]],
                         ids=["gradient-rows", "paths"])
def test_limit_splits_joined(hip_ctx, make):
    b = make()
    print(f"[groups] limits {b.width}x{b.height}", flush=True)
    compare(hip_ctx, b.build(), b.width, b.height)


def test_flushes_that_differ_run_on_their_own(hip_ctx):
    print("[groups] mixed dither", flush=True)
    s = rivehip.generate_stream(2, seed=18, width=640, height=400, draw_count=2600)

    def change(frame):
        frame[-1].dither = 0

    try:
        compare(hip_ctx, s, 640, 400, change)
    finally:
        rivehip.free_stream(s)
