"""Counting and emission take a draw's verbs 64 at a time, one wave per draw.
Paths whose verb counts lie around multiples of 64 (the move and close
included), of lines and cubics mixed with repeated points, as fills, feathered
fills and strokes of every join and cap, with one or many contours, must be
laid out as the oracle lays them out: draw ranges, contours and spans bit for
bit."""
import numpy as np
import pytest

import oracle_binding as ob
import rivehip
from streams import BEVEL, BUTT, CLOCKWISE, EVENODD, MITER, ROUND, ROUND_CAP, SQUARE, StreamBuilder

pytestmark = pytest.mark.gpu


def path_cmds(rng, verbs, w, h, closed):
    cmds = [(0, float(rng.uniform(0, w)), float(rng.uniform(0, h)))]
    for _ in range(verbs):
        r = rng.random()
        if r < .1:
            cmds.append((1, *cmds[-1][-2:]))  # a zero-length line
        elif r < .5:
            cmds.append((1, float(rng.uniform(0, w)), float(rng.uniform(0, h))))
        else:
            cmds.append((4, *(float(v) for v in rng.uniform(0, [w, h, w, h, w, h]))))
    return cmds + ([(5,)] if closed else [])


def check_layout(ctx, b, triangulate=False):
    s = b.build()
    ob.set_interior_triangulation(triangulate)
    try:
        f = ob.OracleFlush(s)
    finally:
        ob.set_interior_triangulation(False)
    t = ctx.target(b.width, b.height)
    ctx.set_interior_triangulation(triangulate)
    try:
        for k in range(f.flush_count):
            assert ctx.render_stream(s, t, max_flushes=k + 1) == f.flush_count
            ctx.sync()
            f.select(k)
            draws = ctx.readback(3).view(rivehip.DRAW)
            od = f.draws()
            assert len(draws) == len(od)
            for name, col in (("path_id", 0), ("tess_location", 1), ("tess_vertex_count", 2)):
                assert np.array_equal(draws[name], od[:, col]), name
            # (a contour without curves has no midpoint: a NaN of either sign)
            c, oc = ctx.readback(1).view(rivehip.CONTOUR), f.get(1).view(rivehip.CONTOUR)
            assert np.array_equal(c["midpoint"], oc["midpoint"], equal_nan=True)
            assert np.array_equal(c["path_id"], oc["path_id"])
            assert np.array_equal(c["vertex_index0"], oc["vertex_index0"])
            assert ctx.readback(0).tobytes() == f.get(0).tobytes()
    finally:
        ctx.set_interior_triangulation(False)
        ctx.free_target(t)
        f.close()


@pytest.mark.parametrize("verbs", [1, 2, 61, 62, 63, 64, 65, 66, 127, 128, 129, 300])
def test_verb_counts_around_a_wave(hip_ctx, verbs):
    print(f"[waves] {verbs} verbs", flush=True)
    rng = np.random.default_rng(verbs)
    w, h = 640, 600
    b = StreamBuilder(w, h)
    for rule in (0, EVENODD):
        b.draw(b.path(path_cmds(rng, verbs, w, h, rule == 0), rule), color=0x80ff0000)
    b.draw(b.path(path_cmds(rng, verbs, w, h, True), CLOCKWISE), color=0x80ff0000, feather=9.0)
    for join in (MITER, ROUND, BEVEL):
        for cap in (BUTT, ROUND_CAP, SQUARE):
            b.draw(b.path(path_cmds(rng, verbs, w, h, bool(rng.random() < .4))), color=0x80ff0000, stroke=7.0, join=join,
                   cap=cap)
    check_layout(hip_ctx, b)


@pytest.mark.parametrize("triangulate", [False, True])
@pytest.mark.parametrize("contours,verbs", [(1, 70), (3, 30), (40, 3), (65, 1), (9, 64)])
def test_contours(hip_ctx, contours, verbs, triangulate):
    print(f"[waves] {contours} contours of {verbs} verbs, triangulate {triangulate}", flush=True)
    rng = np.random.default_rng(contours)
    w, h = 900, 800
    b = StreamBuilder(w, h)
    for stroke in (None, 3.0):
        cmds = sum((path_cmds(rng, verbs, w, h, bool(rng.random() < .5)) for _ in range(contours)), [])
        b.draw(b.path(cmds), color=0x80ff0000, stroke=stroke, join=ROUND, cap=ROUND_CAP)
    check_layout(hip_ctx, b, triangulate)
