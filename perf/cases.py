"""The renderer's workloads: what a program that uses it has it do, each as a
case that can be prepared, run and timed through the public entry points
(rivehip.py over include/rive_hip.h).

Every pass ends with the pixels in host memory, as a program that encodes,
serves or checks its frames needs them: rive_hip_read_pixels into a pinned
buffer that the program keeps (frames, batches, images in their own arrays).
A program keeps one context for its frames; cases whose records stay resident
in a context (a frame flushed again, a captured graph, a batch, the
reference-side binding's buffers) keep a context of their own.

Kinds of case
  frame    a draw stream through RiveRenderer: front end, upload, flush
           (configs 1, 2 and 3 of rive_stream_generate: plain fills; fills,
           strokes, gradients and clips; the same with feathers, advanced
           blends and images), with or without interior triangulation
  resident a frame's logical flushes again from the records in device memory
  graph    the same, captured once in a HIP graph and launched
  batch    many canvases in one flush, from the records in device memory
  serve    timed requests of animated scenes, continuous batching
  spans    the reference's own CPU output: TessVertexSpans, ContourData and
           the DrawBatch list mapped every frame, then a SPANS flush
  png/jpeg an encoded image decoded into a device image with its mip chain
"""
import ctypes
import math
import os
import random
import struct
import sys
import zlib

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "rive-runtime_amd"))

import rivehip  # noqa: E402


def listed():
    return [
        # an icon: the smallest canvas and path count of the batch generator;
        # launches and host waits are all of it
        {"name": "icon_64", "kind": "frame", "config": 1, "width": 64, "height": 64, "draws": 10, "triangulate": False},
        # an illustration: the 1024^2, 200-path frame of the benchmark's first config
        {"name": "art_1024", "kind": "frame", "config": 1, "width": 1024, "height": 1024, "draws": 200,
         "triangulate": False},
        # a laptop-screen frame of mixed content at an odd size, its large
        # fills laid out as outer-cubic patches
        {"name": "patches_1367x767", "kind": "frame", "config": 2, "width": 1367, "height": 767, "draws": 600,
         "triangulate": True},
        # the headline: the 1080p 5000-path frame (six logical flushes), records resident
        {"name": "resident_1080p", "kind": "resident", "config": 2, "width": 1920, "height": 1080, "draws": 5000},
        # a game or kiosk loop: one frame captured and launched again and again
        {"name": "graph_720p", "kind": "graph", "config": 2, "width": 1280, "height": 720, "draws": 1000},
        # soft shadows and blends in a window of odd size
        {"name": "feather_961x541", "kind": "frame", "config": 3, "width": 961, "height": 541, "draws": 700,
         "triangulate": False},
        # the largest: 4K, 20 000 draws with feathers, advanced blends and images
        {"name": "feather_4k", "kind": "frame", "config": 3, "width": 3840, "height": 2160, "draws": 20000,
         "triangulate": False},
        # thumbnails: 48 canvases of 64..1024 px sides and 10..2000 paths in one flush
        {"name": "batch_48", "kind": "batch", "canvases": 48},
        # a render server's queue: 24 requests over 8 animated scenes
        {"name": "serve_24", "kind": "serve", "scenes": 8, "requests": 24},
        # the reference's RenderContext in front of the backend (its own spans, patch batches)
        {"name": "spans_800x601", "kind": "spans", "config": 2, "width": 800, "height": 601, "draws": 500},
        # assets: a screenshot-sized PNG and a photo-sized JPEG
        {"name": "png_1440x901", "kind": "png", "width": 1440, "height": 901},
        {"name": "jpeg_1023x768", "kind": "jpeg", "width": 1023, "height": 768, "subsampled": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes spread over the logarithm of each kind's range,
    frames kept below the largest listed one's draws * pixels."""
    kind = rng.choice(["frame", "frame", "frame", "frame", "resident", "graph", "batch", "serve", "spans",
                       rng.choice(["png", "jpeg"])])
    if kind in ("frame", "resident", "graph", "spans"):
        most = {"frame": (3840, 2160, 20000), "resident": (1920, 1080, 5000), "graph": (1920, 1080, 2000),
                "spans": (1920, 1080, 600)}[kind]
        c = {"kind": kind, "config": rng.choice([1, 2, 3]) if kind == "frame" else rng.choice([1, 2])}
        c["width"] = _log_int(rng, 64, most[0])
        c["height"] = max(48, min(most[1], int(c["width"] * rng.uniform(.5, 1.5))))
        c["draws"] = _log_int(rng, 10, most[2])
        if kind == "frame":
            c["triangulate"] = rng.random() < .2
            if c["config"] == 1:
                c["draws"] = min(c["draws"], 5000)
        return c
    if kind == "batch":
        return {"kind": kind, "canvases": rng.randint(2, 48)}
    if kind == "serve":
        return {"kind": kind, "scenes": rng.randint(1, 8), "requests": rng.randint(1, 32)}
    c = {"kind": kind, "width": _log_int(rng, 33, 1440), "height": _log_int(rng, 33, 1024)}
    if kind == "jpeg":
        c["subsampled"] = rng.random() < .7
    return c


# ---- what a program has in hand before the call

class _Held:
    """Closes what a state owns when the state is dropped."""

    def __init__(self):
        self.close = []

    def __del__(self):
        for f in reversed(self.close):
            f()


_shared = {}


def _context(triangulate=False):
    """The program's context for its frames (one per triangulation setting)."""
    if triangulate not in _shared:
        ctx = rivehip.Context(0)
        ctx.set_interior_triangulation(triangulate)
        _shared[triangulate] = ctx
    return _shared[triangulate]


def _own_context(held):
    ctx = rivehip.Context(0)
    held.close.append(ctx.close)
    return ctx


def _target(held, ctx, w, h):
    t = ctx.target(w, h)
    held.close.append(lambda: ctx.free_target(t))
    return t


def _pinned(n):
    return torch.empty(n, dtype=torch.uint8, pin_memory=True)


def _stream(held, case, seed):
    s = rivehip.generate_stream(case["config"], seed=seed + 1, width=case["width"], height=case["height"],
                                draw_count=case["draws"])
    held.close.append(lambda: rivehip.free_stream(s))
    return s


def batch_sizes(case):
    """(width, height, paths) of a batch's canvases: the same for every seed."""
    rng = random.Random(case["canvases"])
    out = []
    for _ in range(case["canvases"]):
        side, aspect = math.exp(rng.uniform(math.log(64), math.log(1024))), math.exp(rng.uniform(math.log(.5), math.log(2)))
        out.append((max(1, round(side * math.sqrt(aspect))), max(1, round(side / math.sqrt(aspect))),
                    round(math.exp(rng.uniform(math.log(10), math.log(2000))))))
    return out


def serve_sizes(case):
    """(scene, width, height) of the requests: the same for every seed."""
    rng = random.Random(1000 * case["scenes"] + case["requests"])
    return [(rng.randrange(case["scenes"]),) + rng.choice([(256, 256), (512, 512), (1920, 1080)])
            for _ in range(case["requests"])]


def prepare(case, seed):
    held = _Held()
    st = {"held": held, "kind": case["kind"]}
    kind = case["kind"]
    if kind in ("frame", "resident", "graph", "spans"):
        w, h = case["width"], case["height"]
        ctx = _context(case["triangulate"]) if kind == "frame" else _own_context(held)
        st.update(ctx=ctx, stream=_stream(held, case, seed), target=_target(held, ctx, w, h), out=_pinned(w * h * 4),
                  shape=(h, w, 4))
        if kind != "frame":
            ctx.render_stream(st["stream"], st["target"])
            ctx.sync()
            st["frame"] = ctx.last_frame()
        if kind == "graph":
            st["graph"] = ctx.frame_graph(st["frame"], st["target"])
            held.close.append(lambda g=st["graph"]: ctx.frame_graph_destroy(g))
        if kind == "spans":
            st.update(_spans_input(ctx, st["frame"], st["target"]))
    elif kind == "batch":
        sizes = batch_sizes(case)
        ctx = _own_context(held)
        streams = []
        for k, (w, h, n) in enumerate(sizes):
            streams.append(_stream(held, {"config": 1, "width": w, "height": h, "draws": n}, seed * 64 + k))
        st.update(ctx=ctx, targets=[_target(held, ctx, w, h) for w, h, _ in sizes], sizes=sizes,
                  out=_pinned(sum(w * h * 4 for w, h, _ in sizes)))
        ctx.render_streams(streams, st["targets"])
        ctx.sync()
        st["frame"] = ctx.last_frame()
    elif kind == "serve":
        rng = random.Random(seed)
        scenes = []
        for _ in range(case["scenes"]):
            sc = rivehip.Scene(rng.getrandbits(48))
            held.close.append(sc.close)
            scenes.append(sc)
        reqs = [(s, rng.uniform(0.0, 4.0), w, h, 0.0) for s, w, h in serve_sizes(case)]
        out = _pinned(sum(w * h * 4 for _, _, w, h, _ in reqs))
        px, at = {}, 0
        for k, (_, _, w, h, _) in enumerate(reqs):
            px[k] = out.numpy()[at:at + w * h * 4].reshape(h, w, 4)
            at += w * h * 4
        st.update(ctx=_context(), scenes=scenes, requests=reqs, pixels=px, out=out)
    else:
        img = _picture(case["width"], case["height"], 4 if kind == "png" else 3, seed)
        st.update(ctx=_context(),
                  data=_png(img) if kind == "png" else _jpeg(img, 90, 2 if case["subsampled"] else 1))
    return st


def _spans_input(ctx, frame, target):
    """A frame's spans, contours and patch runs per logical flush, as the
    reference's RenderContext writes them (read back from a GEOMETRY flush;
    the PATH, PAINT and gradient records are the ones already resident)."""
    spans, contours, descs, batches = [], [], [], []
    for d in frame:
        ctx.flush(d)
        st = ctx.last_flush_stats()
        s, c = ctx.readback(0).copy(), ctx.readback(1).copy()
        draws = ctx.readback(3).view(rivehip.DRAW)
        first = int(draws["tess_location"].min()) // 8
        end = int((draws["tess_location"] + draws["tess_vertex_count"]).max()) // 8
        b = (rivehip.PatchBatch * 1)()
        b[0].first_patch, b[0].patch_count = first, end - first
        e = rivehip.FlushDesc()
        e.target, e.mode, e.dither = target, rivehip.FLUSH_SPANS, d.dither
        e.load_action, e.clear_color = d.load_action, d.clear_color
        e.path_count, e.contour_count, e.tess_span_count = d.path_count, st.contour_count, st.span_count
        e.tess_vertex_count = st.tess_vertex_count
        e.grad_span_count, e.grad_simple_rows, e.grad_complex_rows = (d.grad_span_count, d.grad_simple_rows,
                                                                      d.grad_complex_rows)
        e.first_path, e.first_paint, e.first_paint_aux = d.first_path, d.first_paint, d.first_paint_aux
        e.first_grad_span = d.first_grad_span
        e.first_tess_span = sum(x.size for x in spans) // rivehip.TESS_SPAN.itemsize
        e.first_contour = sum(x.size for x in contours) // rivehip.CONTOUR.itemsize
        e.patch_batches, e.patch_batch_count = ctypes.cast(b, ctypes.c_void_p), 1
        spans.append(s)
        contours.append(c)
        descs.append(e)
        batches.append(b)
    return {"spans": np.concatenate(spans), "contours": np.concatenate(contours), "descs": descs, "batches": batches}


# ---- one pass

def _read(ctx, target, out):
    rivehip.check(ctx.L.rive_hip_read_pixels(ctx.h, target, out.data_ptr()))


def run(state):
    kind, ctx = state["kind"], state["ctx"]
    if kind in ("png", "jpeg"):
        image = ctx.image_decode(state["data"])
        levels = []
        while True:
            levels.append(ctx.image_read(image, len(levels)))
            if levels[-1].shape[:2] == (1, 1):
                break
        ctx.free_image(image)
        return levels
    if kind == "serve":
        ctx.serve(state["scenes"], state["requests"], 8 << 30, 64, pixels=state["pixels"])
        return state["out"]
    if kind == "batch":
        ctx.flush_frame(state["frame"])
        at = 0
        for t, (w, h, _) in zip(state["targets"], state["sizes"]):
            _read(ctx, t, state["out"][at:at + w * h * 4])
            at += w * h * 4
        return state["out"]
    if kind == "frame":
        ctx.render_stream(state["stream"], state["target"])
    elif kind == "resident":
        ctx.flush_frame(state["frame"], state["target"])
    elif kind == "graph":
        ctx.frame_graph_launch(state["graph"])
    else:
        ctx.upload("tess_span", state["spans"])
        ctx.upload("contour", state["contours"])
        for d in state["descs"]:
            ctx.flush(d)
    _read(ctx, state["target"], state["out"])
    return state["out"].view(state["shape"])


# ---- what a pass cannot do without

def _frame_work(config, w, h, draws):
    # Read: verbs, points (three per cubic; 4-64 cubics a path, 8-32 in config
    # 1; a tenth of the draws of the other configs clip to two 8-cubic paths)
    # and one path, paint and draw record each.  Write: the pixels.  Compute:
    # a src-over blend (four fused multiply-adds) at the pixels a path covers;
    # a random closed path of these configs covers about half of the canvas,
    # a stroke (a fifth of the draws) about a tenth.
    cubics = 20 if config == 1 else 34 + .2 * 8
    covered = .5 if config == 1 else .8 * .5 + .2 * .1
    images = 64 * 256 * 256 * 4 if config == 3 else 0
    return {"bytes": draws * (cubics * 25 + 64 + 8 + 96) + 4 * w * h + images, "flops": 8 * covered * draws * w * h}


def work(case):
    kind = case["kind"]
    if kind in ("frame", "resident", "graph"):
        return _frame_work(case["config"], case["width"], case["height"], case["draws"])
    if kind == "spans":
        # 64 B a span (about one per cubic) in place of the verbs and points
        v = _frame_work(case["config"], case["width"], case["height"], case["draws"])
        v["bytes"] += case["draws"] * (20 if case["config"] == 1 else 35) * 39
        return v
    if kind == "batch":
        parts = [_frame_work(1, w, h, n) for w, h, n in batch_sizes(case)]
    elif kind == "serve":
        # a scene has about 760 paths over at most the square in the request's middle
        parts = [_frame_work(1, min(w, h), min(w, h), 760) for _, w, h in serve_sizes(case)]
        for p, (_, w, h) in zip(parts, serve_sizes(case)):
            p["flops"] *= .1
            p["bytes"] += 4 * (w * h - min(w, h) ** 2)
    else:
        # the encoded bytes (measured: 2.2 a pixel of the PNG, 0.9 of the JPEG),
        # the texels and a third more for the mips; JPEG: a separable 8-point
        # transform and the colour conversion
        px = case["width"] * case["height"]
        mips = 4 * px * 4 / 3
        return {"bytes": (2.2 if kind == "png" else .9) * px + mips, "flops": px * (20 if kind == "png" else 120)}
    return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}


def tolerance(case):
    """Pixels are bytes, quantized after every path: another correct
    implementation rounds a few the other way (the order of a multiply-add,
    a coverage at a tie).  Measured against the CPU implementation of the same
    renderer (the test oracle), as the share of bytes that differ: 0.0005 at
    1024^2 and 1080p, 0.0018 at 640x361, 0.006 at 64x64 (all by 1/255); 0.008
    to 0.022 with feathers; decoded JPEG against 64-bit arithmetic 0.015 to
    0.03.  The limits are four times that where the share is not capped."""
    if case["kind"] == "png":
        return "exact"
    if case["kind"] == "jpeg" or case.get("config") == 3 or case.get("width", 1024) * case.get("height", 1024) < 40000:
        return {"rel": 0.0, "differ": 0.01}
    return {"rel": 0.0, "differ": 0.007}


# ---- image files

def _picture(w, h, channels, seed):
    """Smooth gradients under noise: a screenshot with a photograph's grain (4
    channels), a photograph (3 channels, the grain that survives quality 90)."""
    rng = np.random.default_rng(seed)
    yy, xx = np.mgrid[0:h, 0:w]
    a = 2 * np.pi * rng.random(8)
    base = [128 + 60 * np.sin(xx * (3 + k) / w + a[k]) + 60 * np.cos(yy * (2 + k) / h + a[4 + k]) for k in range(channels)]
    grain = 4 if channels == 4 else 24
    img = np.stack(base, -1) + rng.integers(-grain, grain + 1, (h, w, channels))
    return np.clip(img, 0, 255).astype(np.uint8)


def _png(img):
    h, w, c = img.shape
    rows = img.reshape(h, -1)
    sub = rows.copy()
    sub[:, c:] -= rows[:, :-c]  # filter 1 (Sub)
    raw = np.concatenate([np.ones((h, 1), np.uint8), sub], 1).tobytes()

    def chunk(kind, body):
        return struct.pack(">I", len(body)) + kind + body + struct.pack(">I", zlib.crc32(kind + body) & 0xFFFFFFFF)

    return (b"\x89PNG\r\n\x1a\n" + chunk(b"IHDR", struct.pack(">IIBBBBB", w, h, 8, 6, 0, 0, 0)) +
            chunk(b"IDAT", zlib.compress(raw, 6)) + chunk(b"IEND", b""))


_ZIGZAG = np.array(sorted(range(64), key=lambda i: (i // 8 + i % 8,
                                                    i // 8 if (i // 8 + i % 8) & 1 else i % 8)))
_QUANT = {"y": 8, "c": 17}  # the DC step at quality 50; later ones grow with the frequency


def _dct8():
    x, u = np.mgrid[0:8, 0:8]
    m = np.cos((2 * x + 1) * u * np.pi / 16).T / 2
    m[0] /= math.sqrt(2)
    return m


def _quant(kind, quality):
    i, j = np.mgrid[0:8, 0:8]
    q = _QUANT[kind] * (1 + .45 * (i + j)) * (200 - 2 * quality) / 100
    return np.clip(np.round(q), 1, 255).astype(np.int64)


def _ycc(img):
    r, g, b = (img[..., k].astype(np.float64) for k in range(3))
    y = .299 * r + .587 * g + .114 * b
    return y, (b - y) / 1.772 + 128, (r - y) / 1.402 + 128


def _jpeg_blocks(img, quality, sub):
    """Per component (h = v = its sampling): quantized blocks (by, bx, 8, 8)."""
    h, w = img.shape[:2]
    ph, pw = -h % (8 * sub), -w % (8 * sub)
    out = []
    for k, plane in enumerate(_ycc(img)):
        p = np.pad(plane, ((0, ph), (0, pw)), mode="edge") - 128
        if k and sub == 2:
            p = p.reshape(p.shape[0] // 2, 2, p.shape[1] // 2, 2).mean((1, 3))
        b = p.reshape(p.shape[0] // 8, 8, p.shape[1] // 8, 8).transpose(0, 2, 1, 3)
        f = _dct8() @ b @ _dct8().T
        out.append(np.round(f / _quant("y" if k == 0 else "c", quality)).astype(np.int64))
    return out


def _code(symbols, lengths):
    """Canonical code of the symbols, most frequent first: {symbol: (code, length)} arrays."""
    code, nbits = np.zeros(256, np.int64), np.zeros(256, np.int64)
    at, k = 0, 0
    for n, count in enumerate(lengths, 1):
        for _ in range(count):
            if k < len(symbols):
                code[symbols[k]], nbits[symbols[k]] = at, n
                at, k = at + 1, k + 1
        at <<= 1
    return code, nbits


def _jpeg(img, quality, sub):
    """A baseline JPEG (one interleaved scan, JFIF), chroma halved both ways when sub is 2."""
    h, w = img.shape[:2]
    comps = _jpeg_blocks(img, quality, sub)
    mh, mw = comps[0].shape[0] // sub, comps[0].shape[1] // sub
    # blocks in scan order: an MCU's luma blocks, then one of each chroma
    luma = comps[0].reshape(mh, sub, mw, sub, 64).transpose(0, 2, 1, 3, 4).reshape(mh * mw, sub * sub, 64)
    per = [luma] + [c.reshape(mh * mw, 1, 64) for c in comps[1:]]
    blocks = np.concatenate(per, 1).reshape(-1, 64)[:, _ZIGZAG]
    comp = np.tile(np.concatenate([np.full(p.shape[1], k) for k, p in enumerate(per)]), mh * mw)
    dc = blocks[:, 0].copy()
    for k in range(3):
        dc[comp == k] = np.diff(blocks[comp == k, 0], prepend=0)
    size = lambda v: np.ceil(np.log2(np.abs(v) + 1)).astype(np.int64)  # noqa: E731
    extra = lambda v, s: np.where(v < 0, v + (1 << s) - 1, v)  # noqa: E731
    bl, pos = np.nonzero(blocks[:, 1:])
    pos = pos + 1
    v = blocks[bl, pos]
    prev = np.concatenate([[0], pos[:-1]])
    prev[np.concatenate([[True], bl[1:] != bl[:-1]])[:len(bl)]] = 0
    gap = pos - prev - 1
    zrl = np.repeat(np.arange(len(bl)), gap // 16)
    last = np.zeros(len(blocks), np.int64)
    np.maximum.at(last, bl, pos)
    eob = np.flatnonzero(last < 63)
    # tokens: (order key, symbol, extra bits, their count); DC symbols apart
    s, sd = size(v), size(dc)
    key = np.concatenate([bl * 256 + pos * 2 + 1, bl[zrl] * 256 + pos[zrl] * 2, eob * 256 + 200, np.arange(len(dc)) * 256])
    sym = np.concatenate([(gap % 16) * 16 + s, np.full(len(zrl), 0xF0), np.zeros(len(eob), np.int64), sd])
    val = np.concatenate([extra(v, s), np.zeros(len(zrl) + len(eob), np.int64), extra(dc, sd)])
    cnt = np.concatenate([s, np.zeros(len(zrl) + len(eob), np.int64), sd])
    is_dc = np.arange(len(key)) >= len(key) - len(dc)
    order = np.argsort(key, kind="stable")
    sym, val, cnt, is_dc = sym[order], val[order], cnt[order], is_dc[order]
    tables, codes, nbits = b"", np.zeros(len(sym), np.int64), np.zeros(len(sym), np.int64)
    for cls, which, lengths in ((0, is_dc, [0, 1, 5, 1, 1, 1, 1, 1, 1]),
                                (1, ~is_dc, [0, 2, 1, 3, 3, 2, 4, 3, 5, 5, 4, 4, 0, 0, 1, 125])):
        used, n = np.unique(sym[which], return_counts=True)
        used = used[np.argsort(-n, kind="stable")]
        code, nb = _code(used, lengths)
        codes[which], nbits[which] = code[sym[which]], nb[sym[which]]
        counts = [int((nb[used] == k).sum()) for k in range(1, 17)]
        tables += struct.pack(">HB", 19 + len(used), cls << 4) + bytes(counts) + bytes(used.tolist())
        tables = tables if cls else b"\xff\xc4" + tables + b"\xff\xc4"
    word, length = (codes << cnt) | val, nbits + cnt
    start = np.cumsum(length) - length
    bit = np.arange(int(length.sum())) - np.repeat(start, length)
    bits = (np.repeat(word, length) >> (np.repeat(length, length) - 1 - bit)) & 1
    bits = np.concatenate([bits, np.ones(-len(bits) % 8, np.int64)])
    data = np.packbits(bits.astype(np.uint8)).tobytes().replace(b"\xff", b"\xff\x00")
    head = b"\xff\xd8\xff\xe0" + struct.pack(">H", 16) + b"JFIF\0\x01\x01\0\0\x01\0\x01\0\0"
    for k, name in enumerate("yc"):
        head += b"\xff\xdb" + struct.pack(">HB", 67, k) + bytes(_quant(name, quality).reshape(64)[_ZIGZAG].tolist())
    head += b"\xff\xc0" + struct.pack(">HBHHB", 17, 8, h, w, 3)
    head += bytes([1, sub * 16 + sub, 0, 2, 0x11, 1, 3, 0x11, 1])
    scan = b"\xff\xda" + struct.pack(">HB", 12, 3) + bytes([1, 0, 2, 0, 3, 0, 0, 63, 0])
    return head + tables + scan + data + b"\xff\xd9"


# ---- the same values in 64 bits

def exact(case, seed):
    """Decoded images by plain arithmetic.  A frame has no such value: its
    pixels are defined by what is rounded on the way (vertices to 1/256 px,
    the color to bytes after every path)."""
    if case["kind"] == "png":
        img = _picture(case["width"], case["height"], 4, seed).astype(np.int64)
        t = img[..., :3] * img[..., 3:] + 128
        img[..., :3] = (t + (t >> 8)) >> 8
    elif case["kind"] == "jpeg":
        img = _jpeg_exact(_picture(case["width"], case["height"], 3, seed), 2 if case["subsampled"] else 1)
    else:
        return None
    levels = [img]
    while levels[-1].shape[:2] != (1, 1):
        a = levels[-1]
        h, w = max(a.shape[0] // 2, 1), max(a.shape[1] // 2, 1)
        y, x = 2 * np.arange(h), 2 * np.arange(w)
        y1, x1 = np.minimum(y + 1, a.shape[0] - 1), np.minimum(x + 1, a.shape[1] - 1)
        rows = a[y] + a[y1]
        levels.append((rows[:, x] + rows[:, x1] + 2) >> 2)
    return [lv.astype(np.uint8) for lv in levels]


def _jpeg_exact(img, sub):
    h, w = img.shape[:2]
    planes = []
    for k, q in enumerate(_jpeg_blocks(img, 90, sub)):
        f = q * _quant("y" if k == 0 else "c", 90)
        n = 8 * sub if k else 8  # subsampled chroma: the block's cosine series at twice the points
        x, u = np.mgrid[0:n, 0:8]
        m = np.cos((2 * x + 1) * u * np.pi / (2 * n)) / 2
        m[:, 0] /= math.sqrt(2)
        p = m @ f @ m.T
        planes.append(np.clip(np.round(p.transpose(0, 2, 1, 3).reshape(p.shape[0] * n, -1) + 128), 0, 255)[:h, :w])
    y, cb, cr = planes[0], planes[1] - 128, planes[2] - 128
    rgb = np.stack([y + 1.402 * cr, y - .344136 * cb - .714136 * cr, y + 1.772 * cb], -1)
    rgb = np.clip(np.round(rgb), 0, 255).astype(np.int64)
    return np.concatenate([rgb, np.full((h, w, 1), 255, np.int64)], -1)
