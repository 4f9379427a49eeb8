"""A ContourData record's first vertex may hold any 32-bit index: one beyond the
tessellation reads its last texel, whether it is a little beyond, beyond 2^31
(where it is no signed index) or the largest.  Plain and feathered fills whose
contours wrap to such an index draw the same for all of them."""
import numpy as np
import pytest

import oracle_binding as ob
from streams import CLOCKWISE, StreamBuilder

pytestmark = pytest.mark.gpu


class Edited:
    """An oracle layout with its ContourData records replaced."""

    def __init__(self, f, contours):
        self.f, self.contours = f, contours

    def __getattr__(self, name):
        return getattr(self.f, name)

    def get(self, what):
        return self.contours if what == 1 else self.f.get(what)


@pytest.mark.parametrize("feather", [0.0, 12.0])
def test_first_vertex_beyond_the_tessellation(hip_ctx, feather):
    print(f"[contour-index] {feather}", flush=True)
    b = StreamBuilder(96, 80, clear_color=0xff000000)
    b.draw(b.path([(0, 20, 16), (1, 70, 20), (4, 90, 40, 60, 70, 30, 60), (5,)], CLOCKWISE), color=0xffff8040,
           feather=feather)
    f = ob.OracleFlush(b.build())
    t = hip_ctx.target(96, 80)
    try:
        rows = -(-f.tess_vertex_count // 2048)
        out = []
        for index in (rows * 2048 - 1, rows * 2048, 0x7fffffff, 0x80000000, 0xffffffff):
            c = f.get(1).copy()
            c["vertex_index0"] = index
            ob.OracleFlush.flush_spans_on(Edited(f, c), hip_ctx, t, dither=0)
            out.append(hip_ctx.read_pixels(t, 96, 80))
        for k, px in enumerate(out[1:]):
            assert np.array_equal(out[0], px), k
    finally:
        hip_ctx.free_target(t)
        f.close()
