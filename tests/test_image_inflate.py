"""Inflating and unfiltering a PNG's rows: streams of literals, long runs, matches
at distances below and above a copy's 16 bytes, codes longer than the table's
index, stored and fixed blocks, in sizes around the margins within which symbols
are taken by table steps, for every row filter and pixel size; each must give
back its pixels exactly, and with its last bytes cut off must be refused."""
import numpy as np
import pytest

import rivehip
from test_image_decode import encode_png, expected_rgba


def samples(kind, h, w, ch, rng):
    n = h * w * ch
    if kind == "noise":
        s = rng.integers(0, 256, n)
    elif kind == "run":
        s = np.full(n, 77)
    elif kind == "period":  # matches at short distances
        s = np.tile(rng.integers(0, 256, 7), n // 7 + 1)[:n]
    elif kind == "far":  # matches at long distances
        s = np.tile(rng.integers(0, 256, 1000), n // 1000 + 1)[:n]
    else:  # skewed: rare values get codes longer than 11 bits
        s = np.minimum(rng.geometric(.45, n) - 1, 255)
    return s.reshape(h, w, ch).astype(np.uint8)


@pytest.mark.parametrize("w,h", [(1, 1), (3, 7), (17, 4), (23, 12), (67, 41), (160, 120)])
@pytest.mark.parametrize("kind", ["noise", "run", "period", "far", "skewed"])
def test_streams(kind, w, h):
    rng = np.random.default_rng(w * 1000 + h)
    for ctype, ch in ((0, 1), (2, 3), (4, 2), (6, 4)):
        s = samples(kind, h, w, ch, rng)
        for level in (0, 1, 6, 9):
            data = encode_png(s, ctype, 8, level=level, rng=rng, idat_parts=1 + level % 3)
            assert np.array_equal(rivehip.png_decode(data), expected_rgba(s, ctype, 8)), (ctype, level)
    one = encode_png(s, 6, 8, rng=rng, idat_parts=1)
    with pytest.raises(Exception):
        rivehip.png_decode(one[:-12 - 4 - 5])  # the end of the image data and its checksum
