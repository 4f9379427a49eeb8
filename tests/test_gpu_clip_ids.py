"""Covers hide clip updates only where every update writes a clip ID of its own.
Records that write one ID from two updates, of which one lies hundreds of paths
before an opaque fill over the whole canvas, must draw as if nothing were hidden:
a later draw under that ID shows inside both clips.  The IDs are made equal in
the PAINT records, with the updates in one wave of 64 paths, in neighbouring
ones and far apart, and with IDs of their own in either order."""
import numpy as np
import pytest

import oracle_binding as ob
import rivehip
from streams import StreamBuilder, rect

pytestmark = pytest.mark.gpu
CLIP_UPDATE = 0


class Edited:
    """An oracle layout with its PAINT records replaced."""

    def __init__(self, f, paint):
        self.__dict__["f"], self.__dict__["paint"] = f, paint

    def __getattr__(self, name):
        return getattr(self.f, name)

    def get(self, what):
        return self.paint if what == 3 else self.f.get(what)


def scene(between, after):
    """Two clips on tiles of their own, `between` draws between them and `after`
    from the second to an opaque cover, then red under the second clip."""
    b = StreamBuilder(256, 64, clear_color=0xff000000)
    # (a fifth vertex, so that they are clip paths and not clip rects)
    left, right = (b.path([(0, x, 0), (1, x + 64, 0), (1, x + 64, 64), (1, x, 64), (1, x, 32), (5,)]) for x in (0, 192))
    dot, full = b.path(rect(100, 20, 130, 40)), b.path(rect(0, 0, 256, 64))
    b.draw(full, color=0xff00ff00, clips=(left,))
    for _ in range(between):
        b.draw(dot, color=0x40ffffff)
    b.draw(full, color=0xffffff00, clips=(right,))
    for _ in range(after):
        b.draw(dot, color=0x40ffffff)
    b.draw(full, color=0xff0000ff)
    b.draw(full, color=0xffff0000, clips=(right,))
    return b


@pytest.mark.parametrize("ids", ["same", "descending", "ascending"])
@pytest.mark.parametrize("between,after", [(3, 90), (70, 90), (700, 90), (50, 700)])
def test_updates_of_one_id(hip_ctx, between, after, ids):
    print(f"[clip-ids] {between} {after} {ids}", flush=True)
    b = scene(between, after)
    f = ob.OracleFlush(b.build())
    t = hip_ctx.target(256, 64)
    try:
        paint = f.get(3).copy()
        params, value = paint["params"], paint["value"]
        updates = [i for i in range(1, len(paint)) if (params[i] & 0xf) == CLIP_UPDATE]
        assert len(updates) == 2
        a, z = {"same": (5, 5), "descending": (9, 4), "ascending": (4, 9)}[ids]
        renamed = {int(value[updates[0]] >> 16): a, int(value[updates[1]] >> 16): z}
        for i in range(1, len(paint)):
            if i in updates:
                value[i] = renamed[int(value[i] >> 16)] << 16
            elif params[i] >> 16:
                params[i] = (params[i] & 0xffff) | renamed[int(params[i] >> 16)] << 16
        ob.OracleFlush.flush_spans_on(Edited(f, paint), hip_ctx, t, clear_color=0xff000000, dither=0)
        out = hip_ctx.read_pixels(t, 256, 64)
        red, blue = [255, 0, 0, 255], [0, 0, 255, 255]
        assert (out[:, 192:] == red).all()
        assert (out[:, 64:192] == blue).all()
        assert (out[:, :64] == (red if ids == "same" else blue)).all()
    finally:
        hip_ctx.free_target(t)
        f.close()
