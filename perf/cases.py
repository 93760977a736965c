"""The work this library is used for, as cases that can be timed and compared.

A case is one frame: paths, boxes, images and masks drawn onto one or many
canvases.  Three ways of rendering a frame are covered:

  frame    begin -> calls -> flush / end through the Python API or the native
           scene player: what a program does for a picture it draws once
  replay   a retained frame (a display list that stays on the device) rendered
           again, eagerly or as a captured HIP graph
  batch    many canvases as one frame

Every frame starts by covering its canvas (an opaque paper colour, or a clear
on A8), so a pass does not depend on the pixels the previous one left.
Outputs are the canvases' bytes: whole numbers, fixed by the library's
fixed-point arithmetic, so they are compared exactly.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

import blend2d_amd as B
from blend2d_amd import player, train_cost_model, train_tile_model
from blend2d_amd import scene as S

PRGB32, XRGB32, A8 = 1, 2, 3


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one user-interface widget drawn through the Python API: the smallest
        # call there is, bound by launches and round trips
        {"name": "widget", "kind": "widget", "w": 240, "h": 180, "items": 10, "fmt": PRGB32},
        # thumbnails drawn one after another by a native program, one flush
        # each, and read back
        {"name": "thumbnails", "kind": "thumbs", "count": 12, "paths": 60},
        # a vector drawing of solid polygons kept as a display list and
        # replayed as a HIP graph (bench workload c1)
        {"name": "polygons_512", "kind": "polygons", "w": 512, "h": 512, "n": 1000, "fmt": PRGB32, "graph": True},
        # a full HD picture of 10 000 gradient-filled curves, recorded and
        # rendered by a native program and read back (bench workload c2)
        {"name": "cubics_1080p", "kind": "cubics", "w": 1920, "h": 1080, "n": 10000, "native": True},
        # textured shapes with four blend modes on a 4K canvas, a retained
        # frame (bench workload c3)
        {"name": "patterns_4k", "kind": "patterns", "w": 3840, "h": 2160, "n": 2000, "texture": 512, "graph": False},
        # a quarter of the 4096-canvas glyph frame (half A8, half PRGB32) kept
        # on the device and packed into an atlas after each rendering
        {"name": "glyph_atlas", "kind": "glyphs", "count": 1024, "paths": 200, "native": False},
        # glyph canvases recorded by a native program on its client threads,
        # with the sizing model and the tuned schedule, and read back
        {"name": "glyph_frame", "kind": "glyphs", "count": 256, "paths": 200, "native": True},
        # large canvases with paths of very uneven cost, a retained batch
        # (an eighth of bench workload c5)
        {"name": "uneven_batch", "kind": "uneven", "count": 32, "lo": 1024, "hi": 4096, "paths": 64},
        # translucent full-canvas layers on 4K canvases: pure compositing
        {"name": "layers_4k", "kind": "layers", "count": 4, "w": 3840, "h": 2160, "layers": 3, "fmt": PRGB32},
        # images blitted onto 4K canvases: at integer and fractional origins,
        # scaled, and as tiles of a sprite sheet
        {"name": "blits_4k", "kind": "blits", "count": 4, "w": 3840, "h": 2160, "fmt": PRGB32},
        # a colour and a gradient through full-canvas A8 masks on 4K canvases
        {"name": "masks_4k", "kind": "masks", "count": 4, "w": 3840, "h": 2160, "fmt": PRGB32},
        # gradient backgrounds and panels (linear, radial, conic), dithered
        {"name": "panels_1080p", "kind": "panels", "w": 1920, "h": 1080, "panels": 40, "fmt": PRGB32, "dither": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["widget", "thumbs", "polygons", "cubics", "patterns", "glyphs", "uneven", "layers", "blits",
                       "masks", "panels"])
    fmt = rng.choice([PRGB32, PRGB32, XRGB32, A8])
    if kind == "widget":
        return {"kind": kind, "w": _log(rng, 24, 500), "h": _log(rng, 24, 500), "items": rng.randint(2, 16), "fmt": fmt}
    if kind == "thumbs":
        return {"kind": kind, "count": rng.randint(3, 16), "paths": _log(rng, 4, 200)}
    if kind == "polygons":
        return {"kind": kind, "w": _log(rng, 64, 2000), "h": _log(rng, 64, 2000), "n": _log(rng, 20, 2000), "fmt": fmt,
                "graph": rng.random() < 0.5}
    if kind == "cubics":
        return {"kind": kind, "w": _log(rng, 200, 1920), "h": _log(rng, 200, 1080), "n": _log(rng, 100, 8000),
                "native": rng.random() < 0.5}
    if kind == "patterns":
        return {"kind": kind, "w": _log(rng, 300, 3840), "h": _log(rng, 300, 2160), "n": _log(rng, 30, 2000),
                "texture": rng.choice([61, 256, 333, 512]), "graph": rng.random() < 0.5}
    if kind == "glyphs":
        native = rng.random() < 0.5
        return {"kind": kind, "count": _log(rng, 16, 256 if native else 1024), "paths": _log(rng, 20, 200), "native": native}
    if kind == "uneven":
        return {"kind": kind, "count": rng.randint(2, 32), "lo": _log(rng, 200, 1024), "hi": _log(rng, 1025, 4096),
                "paths": rng.randint(4, 64)}
    if kind == "panels":
        return {"kind": kind, "w": _log(rng, 100, 1920), "h": _log(rng, 100, 1080), "panels": rng.randint(4, 60), "fmt": fmt,
                "dither": rng.random() < 0.5}
    case = {"kind": kind, "count": rng.randint(1, 4), "w": _log(rng, 200, 3840), "h": _log(rng, 200, 2160), "fmt": fmt}
    if kind == "layers":
        case["layers"] = rng.randint(1, 6)
    return case


# ---------------------------------------------------------------------------
# Scenes
# ---------------------------------------------------------------------------

def _papered(sc, value):
    """`sc` behind a call that covers the canvas: an opaque fill, or a clear
    on A8 canvases."""
    head = S.Scene(sc.width, sc.height, sc.format)
    if sc.format == A8:
        head.clear_all()
    else:
        head.fill_all_rgba32(0xFF000000 | value)
    sc.cmds[:0] = head.cmds
    sc.fill_count += 1
    return sc


def _fitted(scenes, lo, hi):
    """The scenes on canvases of sizes (log-uniform between `lo` and `hi`)
    that are the same for every seed, their drawings scaled to them."""
    sizes = np.random.default_rng(len(scenes))
    for sc in scenes:
        w, h = (int(round(lo * (hi / lo) ** sizes.random())) for _ in range(2))
        head = S.Scene(w, h, sc.format)
        head.set_transform([w / sc.width, 0.0, 0.0, h / sc.height, 0.0, 0.0])
        sc.width, sc.height = w, h
        sc.cmds[:0] = head.cmds
    return scenes


def _noise(rng, w, h, fmt=PRGB32):
    if fmt == A8:
        return rng.integers(0, 256, size=(h, w), dtype=np.uint8)
    px = rng.integers(0, 1 << 32, size=(h, w), dtype=np.uint32)
    a = (px >> 24).astype(np.uint32)
    out = px & np.uint32(0xFF000000)
    for s in (0, 8, 16):
        out |= ((((px >> s) & 0xFF) * a + 127) // 255).astype(np.uint32) << np.uint32(s)
    return out


def _smooth_mask(rng, w, h):
    """An A8 mask as a program makes them: soft shapes on a mostly empty
    ground, some of it fully covered."""
    y, x = np.mgrid[0:h, 0:w].astype(np.float32)
    m = np.zeros((h, w), dtype=np.float32)
    for _ in range(4):
        cx, cy = rng.random() * w, rng.random() * h
        r = (0.15 + 0.35 * rng.random()) * max(w, h)
        m = np.maximum(m, 1.6 - 1.6 * np.sqrt((x - cx) ** 2 + (y - cy) ** 2) / r)
    return (np.clip(m, 0.0, 1.0) * 255.0).astype(np.uint8)


def _panel_scene(case, seed):
    """A gradient background and `panels` rectangles, rounded rectangles and
    ellipses filled with gradients."""
    rng = np.random.default_rng(seed)
    w, h = case["w"], case["h"]
    sc = S.Scene(w, h, case["fmt"])
    sc.set_gradient_quality(S.GRADIENT_QUALITY_DITHER if case["dither"] else S.GRADIENT_QUALITY_NEAREST)
    for i in range(case["panels"] + 1):
        pw, ph = (w, h) if i == 0 else (float(rng.uniform(0.05, 0.5) * w), float(rng.uniform(0.05, 0.5) * h))
        x, y = (0.0, 0.0) if i == 0 else (float(rng.uniform(-0.1, 0.9) * w), float(rng.uniform(-0.1, 0.9) * h))
        n = int(rng.integers(2, 6))
        opaque = 0xFF000000 if i == 0 or rng.random() < 0.5 else 0x40000000
        stops = [(k / (n - 1), opaque | int(rng.integers(0, 1 << 32))) for k in range(n)]
        extend = int(rng.integers(0, 3))
        kind = i % 3
        if kind == 0:
            vals = [x, y, x + pw, y + ph * float(rng.random())]
        elif kind == 1:
            vals = [x + pw / 2, y + ph / 2, x + pw / 3, y + ph / 2, max(pw, ph) / 2 + 1.0, 0.0]
        else:
            vals = [x + pw / 2, y + ph / 2, float(rng.uniform(0, 6.28)), 1.0]
        sc.set_fill_style_gradient((S.GRADIENT_LINEAR, S.GRADIENT_RADIAL, S.GRADIENT_CONIC)[kind], vals, stops, extend)
        form = 0 if i == 0 else int(rng.integers(0, 4))
        if i == 0:
            sc.fill_all()
        elif form < 2:
            sc.fill_rect_i(int(x), int(y), max(1, int(pw)), max(1, int(ph)))
        elif form == 2:
            sc.fill_geometry(S.GEOMETRY_ROUND_RECT, (x, y, pw, ph, 8.0, 8.0))
        else:
            sc.fill_path(*S.ellipse_path(x + pw / 2, y + ph / 2, pw / 2, ph / 2))
    return _papered(sc, 0x203040)


def _box_scene(case, rng, seed, k):
    """One canvas of the layers, blits and masks cases."""
    w, h, fmt = case["w"], case["h"], case["fmt"]
    sc = S.Scene(w, h, fmt)
    if case["kind"] == "layers":
        for _ in range(case["layers"]):
            sc.set_fill_style_rgba32((int(rng.integers(16, 240)) << 24) | int(rng.integers(0, 1 << 24)))
            sc.fill_all()
    elif case["kind"] == "blits":
        img = sc.add_image(_noise(rng, w, h, A8 if fmt == A8 else PRGB32), A8 if fmt == A8 else PRGB32)
        half = sc.add_image(_noise(rng, max(1, w // 2), max(1, h // 2)))
        sc.blit_image(S.BLIT_I, img, (0, 0))
        if k % 2 == 0:
            sc.blit_image(S.BLIT_D, half, (w * 0.2 + 0.4, h * 0.2 + 0.3))
        else:
            sc.blit_image(S.BLIT_SCALED_I, half, (w // 8, h // 8, w // 2 + w // 5, h // 2 + h // 5))
        side = max(4, min(w, h) // 12)
        for j in range(24):                # sprites of a sheet
            ax, ay = (j % 6) * (max(1, w // 2) // 8), (j // 6) * (max(1, h // 2) // 8)
            sc.blit_image(S.BLIT_I, half, (int(rng.integers(0, w)), int(rng.integers(0, h))),
                          (ax, ay, min(side, max(1, w // 2) - ax), min(side, max(1, h // 2) - ay)))
    else:
        mask = sc.add_image(_smooth_mask(rng, w, h), A8)
        sc.set_fill_style_rgba32((int(rng.integers(64, 256)) << 24) | int(rng.integers(0, 1 << 24)))
        sc.fill_mask(S.MASK_I, mask, (0, 0))
        if k % 2:
            sc.set_fill_style_gradient(S.GRADIENT_LINEAR, [0.0, 0.0, float(w), float(h)],
                                       [(0.0, 0xC0FF0000 | seed % 255), (1.0, 0x800000FF)])
            sc.fill_mask(S.MASK_I, mask, (w // 7, h // 5), (0, 0, w - w // 7, h - h // 5))
    return _papered(sc, int(rng.integers(0, 1 << 24)))


def _scenes(case, seed):
    kind = case["kind"]
    if kind == "polygons":
        src = S.polygons_scene(seed, case["w"], case["h"], case["n"])
        sc = S.Scene(case["w"], case["h"], case["fmt"])
        sc.cmds, sc.fill_count = src.cmds, src.fill_count
        return [_papered(sc, 0xFFFFFF)]
    if kind == "cubics":
        return [_papered(S.cubic_gradient_scene(seed, case["w"], case["h"], case["n"]), 0)]
    if kind == "patterns":
        return [_papered(S.pattern_shapes_scene(seed, case["w"], case["h"], case["n"], pattern_size=case["texture"]), 0x808080)]
    if kind in ("glyphs", "thumbs"):
        return [_papered(sc, 0xFFFFFF) for sc in _fitted(S.glyph_canvases(seed, case["count"], case["paths"]), 32, 256)]
    if kind == "uneven":
        lo, hi = case["lo"], case["hi"]
        return [_papered(sc, 0xF0F0F0) for sc in _fitted(S.cost_canvases(seed, case["count"], lo, hi, case["paths"]), lo, hi)]
    if kind == "panels":
        return [_panel_scene(case, seed)]
    rng = np.random.default_rng(seed)
    return [_box_scene(case, rng, seed, k) for k in range(case["count"])]


# ---------------------------------------------------------------------------
# A program's side of a frame
# ---------------------------------------------------------------------------

class _Pixels:
    """The pixels of a BLImage where they are, for torch: its rows, or the
    whole buffer (row padding included)."""

    def __init__(self, img, whole=False):
        c = B.ctypes
        ptr, stride = c.c_void_p(), c.c_ssize_t()
        B.lib().bl_amd_image_get_data(img.handle, None, None, None, c.byref(ptr), c.byref(stride))
        shape, strides = ((img.height * stride.value,), (1,)) if whole else (
            (img.height, img.width * img.bpp), (stride.value, 1))
        self.img = img
        self.__cuda_array_interface__ = {"shape": shape, "strides": strides, "typestr": "|u1",
                                         "data": (ptr.value, False), "version": 2}


def _pixels(img, whole=False):
    return torch.as_tensor(_Pixels(img, whole), device="cuda")


class _Canvas:
    """A scene with its device images, and a context that can draw it."""

    def __init__(self, sc, whole=False):
        self.scene = sc
        self.images = []
        for fmt, px in sc.images:
            img = B.BLImage(px.shape[1], px.shape[0], fmt)
            img.upload(px)
            self.images.append(img)
        self.target = B.BLImage(sc.width, sc.height, sc.format)
        self.pixels = _pixels(self.target, whole)
        self.ctx = B.BLContext()

    def record(self):
        self.ctx.begin(self.target)
        errors = B.replay_into(self.ctx, self.scene, self.images)
        if errors:
            raise RuntimeError(f"calls failed: {errors[:4]}")


def _settings(learned=False, graph=False):
    """Process-wide settings of the program: the defaults, or the sizing and
    tile models."""
    B.set_render_schedule(B.SCHEDULE_AUTO)
    B.set_graph_replay(graph)
    if learned:
        B.cost_model_set(train_cost_model.load())
        B.tile_model_set(train_tile_model.load())
        B.set_sizing(B.SIZING_LEARNED)
    else:
        B.set_sizing(B.SIZING_EXACT)
        B.autotune_reset()


def _widget_state(case, seed):
    rng = np.random.default_rng(seed)
    w, h = float(case["w"]), float(case["h"])
    items = []
    for i in range(case["items"]):
        iw, ih = float(rng.uniform(0.1, 0.6) * w), float(rng.uniform(0.08, 0.3) * h)
        x, y = float(rng.uniform(0, w - iw)), float(rng.uniform(0, h - ih))
        color = 0x60000000 | int(rng.integers(0, 1 << 32))
        glyphs = []
        for k in range(4):
            s = max(4.0, min(iw / 5.0, ih * 0.8))
            cmds, vtx = S.glyph_path(rng, s, s)
            glyphs.append((cmds, vtx + np.array([x + 4.0 + k * s, y + (ih - s) / 2])))
        items.append({"box": (x, y, iw, ih), "shadow": 0x40000000, "glyphs": glyphs, "ink": color ^ 0x00FFFFFF,
                      "fill": B.BLGradient(B.GRADIENT_LINEAR, [x, y, x, y + ih],
                                           stops=[(0.0, color), (1.0, 0xFF000000 | int(rng.integers(0, 1 << 24)))])})
    img = B.BLImage(case["w"], case["h"], case["fmt"])
    return {"case": case, "img": img, "pixels": _pixels(img), "ctx": B.BLContext(), "items": items,
            "paper": 0xFFE8E8F0 ^ (seed & 0xFF)}


def _draw_widget(st):
    ctx = st["ctx"]
    ctx.begin(st["img"])
    ctx.clear_all()
    ctx.fill_all(st["paper"])
    for it in st["items"]:
        x, y, w, h = it["box"]
        ctx.fill_rect(x + 1.5, y + 2.0, w, h, it["shadow"])
        ctx.set_fill_style(it["fill"])
        ctx.fill_geometry(B.GEOMETRY_ROUND_RECT, (x, y, w, h, 5.0, 5.0))
        for glyph in it["glyphs"]:
            ctx.fill_path(glyph, rgba32=it["ink"])
    ctx.end()
    return st["pixels"]


def prepare(case, seed):
    kind = case["kind"]
    learned = kind == "glyphs" and case["native"]
    _settings(learned, bool(case.get("graph")))
    if kind == "widget":
        return _widget_state(case, seed)
    scenes = _scenes(case, seed)
    st = {"case": case}
    if kind == "thumbs" or case.get("native"):
        st["frame"] = player.Frame(scenes)
        st["threads"] = 1 if len(scenes) == 1 else max(1, min(16, os.cpu_count() or 1))
        if learned:          # the program tunes its frames' schedule once
            st["frame"].render(player.BATCHED, st["threads"])
            st["frame"].autotune(3)
        return st
    whole = kind == "glyphs"
    st["canvases"] = [_Canvas(sc, whole) for sc in scenes]
    if kind in ("polygons", "cubics", "patterns", "glyphs", "uneven"):
        # retained: recorded and flushed once, then replayed
        st["batch"] = _flush(st["canvases"])
    if whole:
        st["atlas"] = [[c.pixels for c in st["canvases"] if (c.scene.format == A8) == a8] for a8 in (True, False)]
    return st


def _flush(canvases):
    batch = B.BLBatch()
    for c in canvases:
        c.record()
        batch.add(c.ctx)
    batch.flush()
    return batch


def run(st):
    kind = st["case"]["kind"]
    if kind == "widget":
        return _draw_widget(st)
    if "frame" in st:
        frame = st["frame"]
        _, errors, _, r = frame.render(player.PLAIN if kind == "thumbs" else player.BATCHED, st["threads"])
        if r or any(errors):
            raise RuntimeError("the frame failed")
        out = [frame.download(k) for k in range(len(frame.scenes))]
        if len(out) <= 16:
            return out
        return [np.concatenate([p.reshape(-1) for p in out if p.dtype == t]) for t in (np.uint8, np.uint32)]
    if "batch" in st:
        if "atlas" not in st:
            st["batch"].replay()
            return [c.pixels for c in st["canvases"]]
        # the library renders on a stream of its own: the last pass's packing
        # has to have read the canvases before they are rendered again
        torch.cuda.current_stream().synchronize()
        st["batch"].replay()
        return [torch.cat(a) for a in st["atlas"] if a]
    batch = _flush(st["canvases"])
    for c in st["canvases"]:
        c.ctx.end()
    batch.close()
    return [c.pixels for c in st["canvases"]]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    """Canvases written once, images read once, and path vertices (16 bytes)
    and gradient stops (12 bytes) read once, from the distributions that the
    inputs are drawn from.  A pass is integer and byte work with no
    floating-point product to speak of."""
    kind = case["kind"]
    bpp = 1 if case.get("fmt") == A8 else 4
    px = case.get("w", 0) * case.get("h", 0)
    mean = lambda lo, hi: (hi - lo) / math.log(hi / lo)   # of a log-uniform size  # noqa: E731
    if kind == "widget":
        n = px * bpp + case["items"] * (4 * 102 * 16 + 100)
    elif kind in ("glyphs", "thumbs"):
        n = case["count"] * (mean(32, 256) ** 2 * 2.5 + (case["paths"] + 1) / 2 * (102 * 16 + 18))
    elif kind == "polygons":
        n = px * bpp + case["n"] * 7.5 * 16
    elif kind == "cubics":
        n = px * 4 + case["n"] * (32 * 16 + 5 * 12)
    elif kind == "patterns":
        n = px * 4 + case["texture"] ** 2 * 4 + case["n"] * 9 * 16
    elif kind == "uneven":
        n = case["count"] * (mean(case["lo"], case["hi"]) ** 2 * 4 + (case["paths"] + 1) / 2 * 24 * 2 * 16)
    elif kind == "layers":
        n = case["count"] * px * bpp
    elif kind == "blits":
        n = case["count"] * px * (bpp + bpp + 1)
    elif kind == "masks":
        n = case["count"] * px * (bpp + 1)
    else:
        n = px * bpp + case["panels"] * 4 * 12
    return {"bytes": float(n), "flops": 0.0}


def tolerance(case):
    """Bytes, defined by the fixed-point arithmetic of the compositing rules."""
    return "exact"


def exact(case, seed):
    """The outputs are whole bytes that are compared exactly: they have no
    value in 64-bit floating point."""
    return None
