"""Tiles that an opaque fill covers start at the last such fill.  Scenes of
large opaque shapes under every fill rule, mixed with translucent ones,
strokes, gradients and draws under clips that are used again after later
opaque covers (so a tile needs clip updates from before its cover), must
match the oracle, alone and as canvases of one flush."""
import numpy as np
import pytest

import oracle_binding as ob
import rivehip
from streams import BEVEL, CLOCKWISE, EVENODD, NONZERO, StreamBuilder, rect

pytestmark = pytest.mark.gpu


def covered_scene(seed, w=300, h=260, draws=150):
    rng = np.random.default_rng(4000 + seed)
    b = StreamBuilder(w, h, clear_color=0xff303030, dither=seed & 1)

    def blob(rule):
        cx, cy = rng.uniform(0, [w, h])
        r = float(rng.uniform(20, 220))
        if rng.random() < .4:
            return b.path(rect(cx - r, cy - r, cx + r, cy + r, clockwise=bool(rng.random() < .7)), rule)
        k = int(rng.integers(4, 9))
        a = np.sort(rng.uniform(0, 2 * np.pi, k)) * (2 if rng.random() < .3 else 1)  # some wind twice
        pts = [(float(cx + r * np.cos(t)), float(cy + r * np.sin(t))) for t in a]
        return b.path([(0, *pts[0])] + [(1, *p) for p in pts[1:]] + [(5,)], rule)

    clips = [blob(NONZERO) for _ in range(3)]
    for _ in range(draws):
        p = blob([NONZERO, EVENODD, CLOCKWISE][int(rng.integers(0, 3))])
        opaque = rng.random() < .5
        color = int(rng.integers(0, 1 << 24)) | ((255 if opaque else int(rng.integers(60, 255))) << 24)
        kw = {}
        if rng.random() < .35:
            first = int(rng.integers(0, 3))
            kw["clips"] = (clips[first],) if rng.random() < .5 else (clips[first], clips[(first + 1) % 3])
        if rng.random() < .15:
            kw.update(stroke=float(rng.uniform(1, 30)), join=BEVEL)
        elif rng.random() < .15:
            kw["gradient"] = ("linear", 0., 0., float(w), float(h), [(0, color), (1, color ^ 0xffffff)])
        elif rng.random() < .1:
            kw["blend"] = 24  # multiply
        b.draw(p, color=color, **kw)
    return b


def check(out, ref, what):
    d = np.abs(out.astype(np.int32) - ref.astype(np.int32)).max(axis=2)
    assert d.max() <= 8 and (d > 2).mean() <= 1e-3, f"{what}: max {d.max()}, frac>2 {(d > 2).mean()}"


@pytest.mark.parametrize("seed", range(8))
def test_covered_scene_matches_oracle(hip_ctx, seed):
    print(f"[hidden] seed {seed}", flush=True)
    b = covered_scene(seed)
    s = b.build()
    f = ob.OracleFlush(s)
    t = hip_ctx.target(b.width, b.height)
    try:
        ref, _ = f.render()
        hip_ctx.render_stream(s, t)
        out = hip_ctx.read_pixels(t, b.width, b.height)
    finally:
        hip_ctx.free_target(t)
        f.close()
    check(out, ref, f"seed {seed}")


def test_covered_canvases_of_one_flush(hip_ctx):
    print("[hidden] batch", flush=True)
    sizes = [(300, 260), (64, 64), (170, 400)]
    bs = [covered_scene(20 + k, w, h, 60) for k, (w, h) in enumerate(sizes)]
    ss = [b.build() for b in bs]
    ts = [hip_ctx.target(w, h) for w, h in sizes]
    try:
        hip_ctx.render_streams(ss, ts)
        outs = [hip_ctx.read_pixels(t, w, h) for t, (w, h) in zip(ts, sizes)]
        for k, s in enumerate(ss):
            f = ob.OracleFlush(s)
            ref, _ = f.render()
            f.close()
            check(outs[k], ref, f"canvas {k}")
    finally:
        for t in ts:
            hip_ctx.free_target(t)
