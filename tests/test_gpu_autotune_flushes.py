"""The autotuner times all flushes of a frame that runs flush by flush (its draw
records do not follow each other): a heavy first flush and light ones after it
must cost what the first costs alone, up to a factor of two for the clock."""
import pytest

import rivehip
from streams import MITER, StreamBuilder

pytestmark = pytest.mark.gpu


def test_all_flushes_of_a_split_frame_are_timed():
    print("[autotune] split frame", flush=True)
    side = 512
    b = StreamBuilder(side, side)
    p = b.path([(0, 0., 0.), (1, float(side), float(side)), (1, 0., float(side)), (1, float(side), 0.)])
    for k in range(2050):  # 2048 gradient rows fill a flush
        stops = [(0.0, 0x20000000 | k), (0.5, 0x20ff0000), (1.0, 0x200000ff)]
        b.draw(p, stroke=200., join=MITER, gradient=("linear", 0., 0., float(side), 0., stops))
    s = b.build()
    ctx = rivehip.Context(0)
    t = ctx.target(side, side)
    try:
        assert ctx.render_stream(s, t) == 2
        heavy, light = ctx.last_frame()
        frame = [heavy, light, light]
        times = {"heavy": [], "light": []}
        for _ in range(5):
            for name, d in (("heavy", heavy), ("light", light)):
                ctx.flush(d)
                times[name].append(ctx.pass_times()[4])
        alone, last = sorted(times["heavy"])[2], sorted(times["light"])[2]
        assert last < alone / 8
        _, got = ctx.autotune_frame(frame, trials=3)
        print(f"[autotune] {alone} {last} {got}", flush=True)
        assert min(got.values()) > alone / 2
    finally:
        ctx.free_target(t)
        ctx.close()
