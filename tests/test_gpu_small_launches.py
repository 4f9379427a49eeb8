"""Work put into fewer launches: the mip levels an image's blocks make by
themselves (six levels a launch), against the rounded 2x2 means of the level
below; and scans of few values in one workgroup, three at once for a flush's
counts, on either side of its 4096-value steps and of its limit, where a frame's
layout must be the oracle's."""
import numpy as np
import pytest

import rivehip
from streams import StreamBuilder
from test_gpu_counting_waves import check_layout

pytestmark = pytest.mark.gpu


def mips(img):
    levels = [img]
    while max(levels[-1].shape[:2]) > 1:
        s = levels[-1].astype(np.int64)
        h, w = s.shape[:2]
        dh, dw = max(h >> 1, 1), max(w >> 1, 1)
        y0, x0 = np.minimum(2 * np.arange(dh), h - 1), np.minimum(2 * np.arange(dw), w - 1)
        y1, x1 = np.minimum(y0 + 1, h - 1), np.minimum(x0 + 1, w - 1)
        total = s[y0][:, x0] + s[y0][:, x1] + s[y1][:, x0] + s[y1][:, x1]
        levels.append(((total + 2) >> 2).astype(np.uint8))
    return levels


@pytest.mark.parametrize("w,h", [(1, 1), (2, 1), (1, 200), (63, 65), (64, 64), (65, 63), (127, 3), (128, 129),
                                 (333, 190), (1025, 70), (4100, 2)])
def test_mip_chain(hip_ctx, w, h):
    print(f"[mips] {w}x{h}", flush=True)
    img = np.random.default_rng(w * 7 + h).integers(0, 256, (h, w, 4), np.uint8)
    handle = hip_ctx.image(img)
    try:
        for level, want in enumerate(mips(img)):
            assert np.array_equal(hip_ctx.image_read(handle, level), want), level
    finally:
        hip_ctx.free_image(handle)


@pytest.mark.parametrize("n", [1, 63, 1024, 4095, 4096, 4097, 16384, 16385])
def test_scans_of_few_draws(hip_ctx, n):
    print(f"[scans] {n} draws", flush=True)
    b = StreamBuilder(64, 64)
    paths = [b.path([(0, 3, 3), (1, 9 + k, 3), (4, 20, 9, 30 - k, 30, 9, 9), (5,)]) for k in range(5)]
    for k in range(n):
        b.draw(paths[(k * k) % 5], color=0xff000000 | k)
    check_layout(hip_ctx, b)
