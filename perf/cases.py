"""The work this framework is used for, as timed cases.

Every case is one frame (or one batch of frames) as a program has it drawn:
the scene is in hand (packed, and prepared on the device where such a program
draws it more than once), the surface exists, the pre-sizer's weights are
installed; one pass clears the target, draws, and reads the pixels back.
Pixels are bytes defined by the reference's integer rules, so two correct
implementations agree exactly and every tolerance is "exact".

A case is a dict with "kind" (one of KINDS below) and that kind's sizes.
"""
import math

import numpy as np
import torch

from skity_amd import abi, canvas, device, presizer, scenes

_ctx = None


def _context():
    """The program's one context, with the pre-sizer's weights installed."""
    global _ctx
    if _ctx is None:
        if torch.cuda.is_available():
            torch.cuda.init()  # torch's HIP runtime comes up before the library's
        _ctx = device.Context(0)
        params, margin = presizer.load()
        presizer.install(_ctx, params, margin)
    return _ctx


# What each kind stands for:
#   icon      a toolbar icon or a cursor: a few small shapes on a tiny target,
#             recorded afresh (drawn without a prepared scene); the smallest
#             calls, where latency and launches are everything
#   interface an application frame of panels, buttons, separators, progress
#             arcs and avatars, recorded afresh for every frame
#   polygons  plain polygon fills (the generator's workload 1 family)
#   text      a page of glyph-sized outlines drawn as glyph runs
#   curves    fills and strokes of long curved paths (workload 2 family; with
#             4,096 paths it is the benchmark's headline scene)
#   effects   gradient-filled shapes under mask-filter blurs (workload 3 family
#             at screen sizes)
#   picture   a vector illustration: a few hundred large cubic outlines,
#             filled and stroked under a canvas matrix (an SKP's usual content)
#   chart     polylines of many short segments, stroked (plots, map lines)
#   options   every other option used in earnest in one frame: clips, blend
#             modes, colour filters, image shaders, all gradient kinds, on a
#             BGRA target that is not premultiplied
#   batch     many independent canvases of closed outlines drawn by one call
#             (workload 4 family)
KINDS = ("icon", "interface", "polygons", "text", "curves", "effects", "picture", "chart",
         "options", "batch")


def listed():
    return [
        # a 48 px icon of six shapes
        dict(name="icon 48", kind="icon", width=48, height=48, n=6, mode="exact"),
        # a 720p application frame
        dict(name="interface 1280x720", kind="interface", width=1280, height=720, n=420,
             mode="exact"),
        # plain polygons at the reference's example size
        dict(name="polygons 800x600", kind="polygons", n=64, mode="exact"),
        # a dense text page (the benchmark's page has about 17,000 glyphs)
        dict(name="text 2048 learned", kind="text", width=2048, height=2048, n=16900, px=14.0,
             mode="learned"),
        # a caption line on an odd-sized strip
        dict(name="text 701x93", kind="text", width=701, height=93, n=160, px=22.0, mode="exact"),
        # the headline scene, single-pass form
        dict(name="curves 4096 learned", kind="curves", n=4096, mode="learned"),
        # a smaller frame of the same family, plain two-pass form
        dict(name="curves 300 exact", kind="curves", n=300, mode="exact"),
        # gradients and blurred shadows on a laptop screen
        dict(name="effects 1536x960", kind="effects", width=1536, height=960, n=220,
             mode="exact"),
        # an illustration of 305 outlines at 4K
        dict(name="picture 2160 learned", kind="picture", width=3840, height=2160, n=305,
             mode="learned"),
        # plotted lines on an odd-sized target
        dict(name="chart 1921x1083", kind="chart", width=1921, height=1083, n=48, points=1200,
             mode="exact"),
        # all other options, BGRA and not premultiplied
        dict(name="options 1000x700", kind="options", width=1000, height=700, n=260,
             mode="exact"),
        # twelve canvases by one call
        dict(name="batch 12 learned", kind="batch", canvases=12, n=260, mode="learned"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    mode = rng.choice(("exact", "learned"))
    if kind == "icon":
        return dict(kind=kind, width=_log_int(rng, 9, 160), height=_log_int(rng, 9, 160),
                    n=rng.randint(1, 16), mode=mode)
    if kind == "interface":
        return dict(kind=kind, width=_log_int(rng, 200, 2600), height=_log_int(rng, 150, 1600),
                    n=_log_int(rng, 20, 1500), mode=mode)
    if kind == "polygons":
        return dict(kind=kind, n=_log_int(rng, 4, 900), mode=mode)
    if kind == "text":
        return dict(kind=kind, width=_log_int(rng, 120, 2600), height=_log_int(rng, 40, 2200),
                    n=_log_int(rng, 20, 18000), px=rng.uniform(7.0, 60.0), mode=mode)
    if kind == "curves":
        # the plain form walks its longest path twice: few paths cost it as much
        return dict(kind=kind, n=_log_int(rng, 6, 1800 if mode == "learned" else 300), mode=mode)
    if kind == "effects":
        return dict(kind=kind, width=_log_int(rng, 200, 2100), height=_log_int(rng, 200, 1500),
                    n=_log_int(rng, 4, 500), mode=mode)
    if kind == "picture":
        return dict(kind=kind, width=_log_int(rng, 256, 4096), height=_log_int(rng, 256, 2800),
                    n=_log_int(rng, 20, 700), mode=mode)
    if kind == "chart":
        return dict(kind=kind, width=_log_int(rng, 200, 2600), height=_log_int(rng, 120, 1600),
                    n=_log_int(rng, 2, 90), points=_log_int(rng, 12, 2400), mode=mode)
    if kind == "options":
        return dict(kind=kind, width=_log_int(rng, 64, 1700), height=_log_int(rng, 64, 1300),
                    n=_log_int(rng, 10, 500), mode=mode)
    return dict(kind="batch", canvases=rng.randint(2, 24), n=_log_int(rng, 20, 500), mode=mode)


# ---- scenes -----------------------------------------------------------------

def _rgba(r, lo_alpha=0.3):
    return tuple(float(v) for v in r.integers(0, 256, 3) / 255.0) + (
        float(r.integers(int(lo_alpha * 255), 256) / 255.0),)


def _gradient(r, x, y, size, kinds=(abi.GRADIENT_LINEAR, abi.GRADIENT_RADIAL)):
    g = abi.Gradient()
    g.type = int(r.choice(kinds))
    g.tile_mode = int(r.integers(0, 3))
    g.color_count = int(r.integers(2, 9))
    g.has_offsets = 1
    for i, o in enumerate(np.sort(r.random(g.color_count))):
        g.offsets[i] = float(o)
        for c in range(4):
            g.colors[i][c] = float(r.random()) if c < 3 else float(0.4 + 0.6 * r.random())
    g.points[0], g.points[1] = x, y
    if g.type == abi.GRADIENT_LINEAR:
        g.points[2], g.points[3] = x + size, y + 0.5 * size
    elif g.type == abi.GRADIENT_RADIAL:
        g.radius[0] = max(0.6 * size, 1.0)
    elif g.type == abi.GRADIENT_SWEEP:
        g.radius[0], g.radius[1] = -0.125, 1.0 / 0.75
    else:  # two-point conical
        g.points[2], g.points[3] = x + 0.3 * size, y + 0.2 * size
        g.radius[0], g.radius[1] = max(0.1 * size, 0.5), max(0.8 * size, 1.0)
    g.local_matrix[0] = g.local_matrix[4] = 1.0
    return g


def _round_rect(p, l, t, r, b, rad):
    """A rounded rectangle as line and conic verbs."""
    w = canvas.FLOAT_ROOT2_OVER2
    p.move_to(l + rad, t).line_to(r - rad, t).conic_to(r, t, r, t + rad, w)
    p.line_to(r, b - rad).conic_to(r, b, r - rad, b, w)
    p.line_to(l + rad, b).conic_to(l, b, l, b - rad, w)
    p.line_to(l, t + rad).conic_to(l, t, l + rad, t, w)
    return p.close()


def _icon(case, r):
    w, h = case["width"], case["height"]
    cv = canvas.Canvas(w, h)
    s = min(w, h)
    for i in range(case["n"]):
        p, paint = canvas.Path(), canvas.Paint(_rgba(r))
        x, y, q = r.uniform(0.1, 0.9) * w, r.uniform(0.1, 0.9) * h, r.uniform(0.1, 0.45) * s
        k = i % 3
        if k == 0:
            _round_rect(p, x - q, y - q, x + q, y + q, 0.3 * q)
        elif k == 1:
            p.add_circle(x, y, q)
        else:
            p.move_to(x - q, y).line_to(x, y + q).line_to(x + q, y - q)
            paint.set_style(abi.STYLE_STROKE).set_stroke_width(1.0 + 0.06 * s)
            paint.set_stroke_cap(abi.CAP_ROUND).set_stroke_join(abi.JOIN_ROUND)
        cv.draw_path(p, paint)
    return cv


def _interface(case, r):
    w, h = case["width"], case["height"]
    cv = canvas.Canvas(w, h)
    cv.draw_paint(canvas.Paint((0.96, 0.96, 0.97, 1.0)))
    for i in range(case["n"]):
        p, paint = canvas.Path(), canvas.Paint(_rgba(r))
        x, y = r.uniform(0, w), r.uniform(0, h)
        bw, bh = r.uniform(20, 0.25 * w + 21), r.uniform(10, 60)
        k = int(r.integers(0, 6))
        if k <= 1:
            _round_rect(p, x, y, x + bw, y + bh, 6.0)
            if k:
                paint.set_gradient(_gradient(r, x, y, bw))
        elif k == 2:
            p.add_rect(math.floor(x), math.floor(y), math.floor(x + bw), math.floor(y + 1))
        elif k == 3:
            p.add_circle(x, y, r.uniform(4, 28))
        elif k == 4:
            _round_rect(p, x, y, x + bw, y + bh, 4.0)
            paint.set_style(abi.STYLE_STROKE).set_stroke_width(1.5)
        else:
            p.move_to(x, y).cubic_to(x + 15, y - 25, x + 35, y + 25, x + 50, y)
            paint.set_style(abi.STYLE_STROKE).set_stroke_width(3.0)
            paint.set_stroke_cap(abi.CAP_ROUND)
        cv.draw_path(p, paint)
    return cv


def _glyph(r):
    """An outline in a unit em with the verb counts of a text face's glyphs
    (a contour or two of lines and quads, 6 to 57 verbs)."""
    p = canvas.Path()
    for c in range(int(r.integers(1, 3))):
        m = int(r.integers(4, 27))
        cx, cy = r.uniform(0.25, 0.35), r.uniform(-0.4, -0.3)
        rad = (0.30 if c == 0 else 0.14) * r.uniform(0.8, 1.2)
        th = np.linspace(0, 2 * math.pi, m + 1) * (1 if c == 0 else -1)
        jit = r.uniform(0.75, 1.25, m + 1)
        jit[m] = jit[0]
        xs, ys = cx + rad * jit * np.cos(th), cy + 1.2 * rad * jit * np.sin(th)
        p.move_to(xs[0], ys[0])
        for i in range(m):
            if r.random() < 0.45:
                p.line_to(xs[i + 1], ys[i + 1])
            else:
                mx, my = 0.5 * (xs[i] + xs[i + 1]), 0.5 * (ys[i] + ys[i + 1])
                p.quad_to(cx + 1.15 * (mx - cx), cy + 1.15 * (my - cy), xs[i + 1], ys[i + 1])
        p.close()
    return p


def _text(case, r):
    w, h, px = case["width"], case["height"], case["px"]
    cv = canvas.Canvas(w, h)
    cv.draw_paint(canvas.Paint((1.0, 1.0, 1.0, 1.0)))
    face = [_glyph(r) for _ in range(64)]
    per_line = max(1, int(w / (0.6 * px)))
    lines = -(-case["n"] // per_line)
    step = max(0.5, (h - 0.2 * px) / lines)
    left = case["n"]
    for line in range(lines):
        k = min(per_line, left)
        left -= k
        cv.save()
        cv.translate(0.0, 0.9 * min(step, px) + line * step)
        cv.scale(px, px)
        if line % 29 == 28:
            cv.rotate(1.5)
        paint = canvas.Paint(_rgba(r, 0.7))
        if line % 31 == 30:
            paint.set_style(abi.STYLE_STROKE).set_stroke_width(0.06)
        cv.draw_glyphs([face[int(g)] for g in r.integers(0, len(face), k)],
                       [0.6 * i for i in range(k)], [0.0] * k, paint)
        cv.restore()
    return cv


def _blob(p, r, cx, cy, rad, anchors, wobble=0.35):
    th = np.linspace(0, 2 * math.pi, anchors + 1)
    m = rad * r.uniform(1 - wobble, 1 + wobble, anchors + 1)
    m[anchors] = m[0]
    xs, ys = cx + m * np.cos(th), cy + m * np.sin(th)
    p.move_to(xs[0], ys[0])
    for i in range(anchors):
        dx, dy = xs[i + 1] - xs[i], ys[i + 1] - ys[i]
        o1, o2 = r.uniform(-0.3, 0.3, 2)
        p.cubic_to(xs[i] + dx / 3 - o1 * dy, ys[i] + dy / 3 + o1 * dx,
                   xs[i] + 2 * dx / 3 - o2 * dy, ys[i] + 2 * dy / 3 + o2 * dx,
                   xs[i + 1], ys[i + 1])
    return p.close()


def _effects(case, r):
    w, h = case["width"], case["height"]
    cv = canvas.Canvas(w, h)
    styles = (abi.BLUR_NORMAL,) * 5 + (abi.BLUR_SOLID, abi.BLUR_OUTER, abi.BLUR_INNER)
    for i in range(case["n"]):
        p, paint = canvas.Path(), canvas.Paint(_rgba(r))
        rad = math.exp(r.uniform(math.log(8), math.log(0.3 * min(w, h))))
        x, y = r.uniform(0, w), r.uniform(0, h)
        _blob(p, r, x, y, rad, 4)
        paint.set_gradient(_gradient(r, x - rad, y - rad, 2 * rad, (
            abi.GRADIENT_LINEAR, abi.GRADIENT_RADIAL, abi.GRADIENT_SWEEP)))
        if i % 4:
            sigma = r.uniform(1.0, 32.0)
            paint.set_blur((sigma - 0.5) / 0.57735, int(r.choice(styles)))
        cv.draw_path(p, paint)
    return cv


def _picture(case, r):
    w, h = case["width"], case["height"]
    cv = canvas.Canvas(w, h)
    cv.draw_paint(canvas.Paint((1.0, 1.0, 1.0, 1.0)))
    # drawn in a 1,000-unit space, as an SKP's own matrix scales it up
    s = max(w, h) / 1000.0
    cv.scale(s, s)
    cv.rotate(3.0)
    for i in range(case["n"]):
        p, paint = canvas.Path(), canvas.Paint(_rgba(r, 0.6))
        rad = math.exp(r.uniform(math.log(5), math.log(330)))
        _blob(p, r, r.uniform(0, 1000), r.uniform(0, 1000 * h / max(w, h)), rad,
              int(r.integers(3, 30)))
        k = i % 5
        if k >= 3:
            paint.set_style(abi.STYLE_STROKE if k == 3 else abi.STYLE_STROKE_AND_FILL)
            paint.set_stroke_width(r.uniform(0.3, 4.0))
        if i % 7 == 0:
            p.fill_type = abi.FILL_EVEN_ODD
        cv.draw_path(p, paint)
    return cv


def _chart(case, r):
    w, h, m = case["width"], case["height"], case["points"]
    cv = canvas.Canvas(w, h)
    cv.draw_paint(canvas.Paint((1.0, 1.0, 1.0, 1.0)))
    for i in range(case["n"]):
        p, paint = canvas.Path(), canvas.Paint(_rgba(r, 0.6))
        xs = np.linspace(0.03 * w, 0.97 * w, m + 1)
        ys = h * (i + 0.5) / case["n"] + np.cumsum(r.normal(0, 0.25 * h / math.sqrt(m), m + 1))
        if i % 3 == 2:  # a map line: it turns around instead of running right
            th = np.cumsum(r.normal(0, 0.35, m + 1))
            d = 2.5 * max(w, h) / m
            xs = r.uniform(0, w) + np.cumsum(d * np.cos(th))
            ys = r.uniform(0, h) + np.cumsum(d * np.sin(th))
        p.move_to(xs[0], ys[0])
        for x, y in zip(xs[1:], ys[1:]):
            p.line_to(x, y)
        paint.set_style(abi.STYLE_STROKE).set_stroke_width(float(r.uniform(0.8, 5.0)))
        paint.set_stroke_join(int(r.integers(0, 3))).set_stroke_cap(int(r.integers(0, 3)))
        cv.draw_path(p, paint)
    return cv


def _options(case, r):
    w, h = case["width"], case["height"]
    cv = canvas.Canvas(w, h)
    cv.draw_paint(canvas.Paint((0.9, 0.95, 1.0, 0.8)))
    image = r.integers(0, 256, (61, 87, 4)).astype(np.uint8)
    blends = [abi.BLEND_SRC_OVER] * 4 + [abi.BLEND_SRC, abi.BLEND_SRC_ATOP, abi.BLEND_DST_OVER,
                                         abi.BLEND_XOR, abi.BLEND_PLUS, abi.BLEND_MODULATE,
                                         abi.BLEND_SCREEN, abi.BLEND_SOFT_LIGHT,
                                         abi.BLEND_DST_OUT]
    for i in range(case["n"]):
        p, paint = canvas.Path(), canvas.Paint(_rgba(r))
        x, y = r.uniform(0, w), r.uniform(0, h)
        rad = math.exp(r.uniform(math.log(4), math.log(0.35 * min(w, h))))
        if i % 2:
            _blob(p, r, x, y, rad, int(r.integers(3, 12)))
        else:
            _round_rect(p, x - rad, y - 0.6 * rad, x + rad, y + 0.6 * rad, 0.2 * rad)
        paint.set_blend_mode(int(r.choice(blends)))
        k = i % 6
        if k == 0:
            paint.set_gradient(_gradient(r, x - rad, y - rad, 2 * rad, (
                abi.GRADIENT_LINEAR, abi.GRADIENT_RADIAL, abi.GRADIENT_CONICAL)))
        elif k == 1:
            paint.set_image_shader(image, abi.ALPHA_UNPREMUL, int(r.integers(0, 2)),
                                   int(r.integers(0, 4)), int(r.integers(0, 4)),
                                   (1.3, 0.2, x, -0.1, 0.9, y))
        elif k == 2:
            paint.set_color_filter(canvas.matrix_color_filter(
                [0.3, 0.6, 0.1, 0, 0, 0.2, 0.7, 0.1, 0, 0, 0.3, 0.3, 0.4, 0, 0, 0, 0, 0, 1, 0]))
        elif k == 3:
            paint.set_style(abi.STYLE_STROKE_AND_FILL).set_stroke_width(2.5)
        if i % 5 == 4:
            cv.save()
            cv.clip_rect(x - 0.7 * rad, y - 0.7 * rad, x + 0.9 * rad, y + 0.5 * rad)
            cv.draw_path(p, paint)
            cv.restore()
        else:
            cv.save()
            cv.rotate(float(r.uniform(-20, 20)), x, y)
            cv.draw_path(p, paint)
            cv.restore()
    return cv


_RECORDED = {"icon": _icon, "interface": _interface, "text": _text, "effects": _effects,
             "picture": _picture, "chart": _chart, "options": _options}
_FRESH = ("icon", "interface")  # drawn from the packed scene, without a prepared one
_GENERATED = {"polygons": 1, "curves": 2}
_MODES = {"exact": abi.MODE_EXACT, "learned": abi.MODE_LEARNED}
_SIDES = (256, 512, 512, 1024)


class _State:
    pass


def _target(case, ctx, width, height):
    if case["kind"] == "options":
        return device.Surface(ctx, width, height, abi.ALPHA_UNPREMUL, abi.COLOR_BGRA)
    return device.Surface(ctx, width, height)


def prepare(case, seed):
    ctx = _context()
    st = _State()
    st.kind, st.mode = case["kind"], _MODES[case["mode"]]
    r = np.random.default_rng(seed)
    if st.kind == "batch":
        st.batch = device.Batch(ctx)
        st.surfaces = []
        for i in range(case["canvases"]):
            side = _SIDES[i % len(_SIDES)]
            sc = scenes.outlines(int(r.integers(1, 1 << 62)), side, 0, case["n"], -5.0, -1.0)
            su = device.Surface(ctx, side, side)
            st.batch.add(su, device.Prepared(ctx, sc.scene))
            st.surfaces.append(su)
        return st
    if st.kind in _GENERATED:
        st.scene = scenes.generate(_GENERATED[st.kind], n_paths=case["n"],
                                   seed=int(r.integers(1, 1 << 62)))
    else:
        st.scene = _RECORDED[st.kind](case, r).scene()
    st.surface = _target(case, ctx, st.scene.width, st.scene.height)
    st.what = st.scene.scene
    if st.kind not in _FRESH:
        st.what = device.Prepared(ctx, st.scene.scene)
    return st


def run(state):
    if state.kind == "batch":
        for su in state.surfaces:
            su.clear(0)
        state.batch.draw(mode=state.mode)
        return [su.read() for su in state.surfaces]
    state.surface.clear(0)
    state.surface.draw(state.what, mode=state.mode)
    return state.surface.read()


# ---- what a pass cannot do without ------------------------------------------

def _size(case):
    if case["kind"] == "polygons":
        return 800, 600
    if case["kind"] == "curves":
        return 2048, 2048
    return case["width"], case["height"]


# points and verbs of a typical draw of each kind, in bytes (8 per point, 1 per
# verb, 32 for the draw itself)
_DRAW_BYTES = {"icon": 150, "interface": 140, "polygons": 200, "text": 330, "curves": 2600,
               "effects": 200, "picture": 450, "options": 250, "batch": 23000}


def work(case):
    """The geometry read once, the target's pixels written once and read back
    once; for a blurred draw its layer besides."""
    kind = case["kind"]
    if kind == "batch":
        px = sum(_SIDES[i % len(_SIDES)] ** 2 for i in range(case["canvases"]))
        return {"bytes": 8.0 * px + _DRAW_BYTES[kind] * case["n"] * case["canvases"], "flops": 0.0}
    w, h = _size(case)
    n = case["n"]
    per = 41 + 9 * case["points"] if kind == "chart" else _DRAW_BYTES[kind]
    out = {"bytes": 8.0 * w * h + per * n, "flops": 0.0}
    if kind == "effects":  # three draws of four are blurred; a mean layer of 0.03 of the target
        out["bytes"] += 0.75 * n * 0.03 * w * h * 8
    return out


def tolerance(case):
    return "exact"


def exact(case, seed):
    """Pixels come from integer rules; they have no 64-bit value of their own."""
    return None
