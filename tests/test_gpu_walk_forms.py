"""GPU parity at the edges of the walk's forms and of the composite's.

The walk keeps 64 edges per wave or slot, takes rows of plain edges several at
a time, marks tiles that a path covers whole without a plane, and runs with or
without row bands and a count pass; the composite has a form for covers of one
colour.  All of it is whole-number arithmetic: the tolerance is none.
"""
import numpy as np
import pytest

from oracle import oracle_py as O
from skity_amd import abi, device, presizer
from skity_amd.canvas import Canvas, Paint, Path, blend_color_filter

from helpers import diff_report

pytestmark = pytest.mark.gpu

# (mode, band rows, smallest banded bound): the default exact form, the counted
# one with short bands, and the learned form with default bands and all banded
FORMS = [(abi.MODE_EXACT, 0, 0), (abi.MODE_EXACT, 16, 0), (abi.MODE_LEARNED, 0, 0),
         (abi.MODE_LEARNED, 32, -1)]


@pytest.fixture(scope="module")
def ctx():
    c = device.Context(0)
    presizer.install(c, *presizer.load())
    yield c
    c.close()


def check(ctx, sc, name):
    want = O.render(sc.scene, sc.width, sc.height)
    counts = set()
    for mode, rows, least in FORMS:
        surf = device.Surface(ctx, sc.width, sc.height)
        print(f"{name}: mode {mode}, band rows {rows}", flush=True)
        surf.draw(sc.scene, mode=mode, band_rows=rows, band_min_edges=least)
        got, st = surf.read(), surf.stats()
        surf.close()
        assert diff_report(got, want) == (0, 0), (mode, rows)
        counts.add((st["max_active"], st["blends"], st["pixels"]))
    assert len(counts) == 1  # the forms agree on what was walked and blended


def spikes(p, x, y, n, height, spread):
    """n spikes (2 n edges and two of the base); their tips lie on `spread`
    different heights, so that n / spread edges start in one row."""
    p.move_to(x - 1.25, y + height)
    for i in range(n):
        p.line_to(x + 2.6 * i, y + 0.6 + (i % spread))
        p.line_to(x + 2.6 * i + 1.3, y + height - (i % 3))
    p.close()
    return p


# 64 .. 1026 active edges: either side of 1, 2, 4, 8 and 16 waves of 64, and of
# the 16 and 64 edges that start at once
@pytest.mark.parametrize("n,spread", [(31, 1), (31, 7), (32, 7), (63, 3), (64, 1), (127, 7),
                                      (128, 1), (255, 5), (256, 2), (511, 1), (512, 7)])
def test_lists_at_the_edges_of_waves(ctx, n, spread):
    w = int(2.6 * n) + 40
    c = Canvas(w, 151)
    c.draw_path(spikes(Path(), 9.3, 12.4, n, 121.5, spread), Paint((0.3, 0.6, 0.9, 0.8)))
    c.draw_path(spikes(Path(), 4.1, 131.2, 5, 40.0, 2), Paint((0.9, 0.2, 0.1, 1.0)))
    check(ctx, c.scene(), f"{n} spikes")


@pytest.mark.parametrize("w,h", [(1, 1), (15, 17), (16, 16), (33, 64), (65, 65), (130, 127)])
def test_plain_rows_and_solid_tiles(ctx, w, h):
    """Straight edges over 1 to all rows, from and to every part of a pixel
    row, inside, across and outside the canvas."""
    rng = np.random.default_rng(1000 * w + h)
    c = Canvas(w, h)
    for i in range(24):
        paint = Paint((0.1 * (i % 9), 0.7, 0.04 * i, (1.0, 0.55, 0.0, 1.0)[i % 4]))
        if i % 5 == 4:
            paint.set_blend_mode((abi.BLEND_SRC, abi.BLEND_CLEAR, abi.BLEND_DST_IN)[i % 3])
        l, r = np.sort(rng.uniform(-0.5 * w - 2, 1.5 * w + 2, 2))
        t, b = np.sort(rng.uniform(-0.5 * h - 2, 1.5 * h + 2, 2))
        if i % 6 == 1:  # whole pixels
            l, t, r, b = np.floor(l), np.floor(t), np.ceil(r), np.ceil(b)
        if i % 6 == 3:  # the whole canvas and more
            l, t, r, b = -3.5, -2.25, w + 4.75, h + 3.5
        lean = rng.uniform(-0.3, 0.3) * (r - l) if i % 2 else 0.0
        p = Path().move_to(l + lean, t).line_to(r, t).line_to(r - lean, b).line_to(l, b).close()
        if i % 4 == 2:  # a hole
            p.add_rect(l + 0.3 * (r - l), t + 0.2 * (b - t), l + 0.6 * (r - l), b - 0.3, ccw=True)
            p.fill_type = abi.FILL_EVEN_ODD
        c.draw_path(p, paint)
    check(ctx, c.scene(), f"{w} x {h}")


@pytest.mark.parametrize("filtered", [False, True])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
def test_covers_of_one_colour(ctx, n, filtered):
    """n paths on every tile (the composite takes 64 at a time), of alpha 0,
    1, 254, 255 and between, beside ones that take the general form."""
    c = Canvas(50, 37)
    for i in range(n):
        a = (255, 128, 1, 254, 0)[i % 5]
        paint = Paint(((37 * i % 256) / 255, (91 * i % 256) / 255, 0.5, a / 255))
        if i % 16 == 7:
            paint.set_blend_mode(abi.BLEND_XOR)
        if filtered and i % 8 == 2:
            paint.set_color_filter(blend_color_filter(0x8040C0FF, abi.BLEND_SRC_ATOP))
        p = Path().add_oval(-9.7 + 0.2 * i, -5.1, 55.3, 40.2 - 0.15 * i)
        if i % 3 == 1:
            p = Path().add_rect(0.25 * (i % 40), -1, 49.5, 38)
        c.draw_path(p, paint)
    sc = c.scene()
    check(ctx, sc, f"{n} paths")
    for alpha, colour in ((abi.ALPHA_UNPREMUL, abi.COLOR_RGBA),
                          (abi.ALPHA_PREMUL, abi.COLOR_BGRA)):
        surf = device.Surface(ctx, sc.width, sc.height, alpha, colour)
        surf.draw(sc.scene)
        got = surf.read()
        surf.close()
        want = O.render_ex(sc.scene, sc.width, sc.height, alpha, colour)
        assert diff_report(got, want) == (0, 0)


@pytest.mark.parametrize("n", [255, 256, 1024, 1025])
def test_many_paths(ctx, n):
    """Small paths, rectangles and whole-canvas draws on two targets of one
    batch: either side of the number of jobs from which the composite scans by
    tile row, and of the 1,024 jobs that a pass over them takes."""
    rng = np.random.default_rng(n)
    scs = []
    for w, h in ((70, 150), (33, 49)):
        c = Canvas(w, h)
        for i in range(n if w == 70 else 40):
            paint = Paint((*rng.uniform(0, 1, 3), rng.uniform(0.2, 1.0)))
            if i % 97 == 5:
                c.draw_paint(paint)
                continue
            x, y, s = rng.uniform(-10, w + 10), rng.uniform(-10, h + 10), rng.uniform(0.5, 9)
            c.draw_path(Path().add_circle(x, y, s) if i % 3 else
                        Path().add_rect(x, y, x + s, y + 4 * s), paint)
        scs.append(c.scene())
    surfs = [device.Surface(ctx, sc.width, sc.height) for sc in scs]
    preps = [device.Prepared(ctx, sc.scene) for sc in scs]
    batch = device.Batch(ctx)
    for su, pr in zip(surfs, preps):
        batch.add(su, pr)
    for mode in (abi.MODE_EXACT, abi.MODE_LEARNED):
        print(f"{n} paths, mode {mode}", flush=True)
        for su in surfs:
            su.clear(0)
        batch.draw(mode=mode)
        for su, sc in zip(surfs, scs):
            assert diff_report(su.read(), O.render(sc.scene, sc.width, sc.height)) == (0, 0)
    batch.close()
    for x in surfs + preps:
        x.close()


@pytest.mark.parametrize("join", [abi.JOIN_MITER, abi.JOIN_ROUND, abi.JOIN_BEVEL])
def test_runs_of_lines(ctx, join):
    """Stroked polylines either side of the shortest run that lanes share, of a
    wave's 64 lines and of a chunk's 128 calls."""
    rng = np.random.default_rng(join)
    c = Canvas(260, 190)
    for i, n in enumerate((1, 2, 3, 4, 63, 64, 65, 66, 127, 128, 129, 130, 300)):
        paint = Paint((*rng.uniform(0, 1, 3), 0.7))
        paint.set_style(abi.STYLE_STROKE).set_stroke_width(float(rng.uniform(0.4, 6)))
        paint.set_stroke_join(join).set_stroke_cap(i % 3)
        p = Path().move_to(130, 95)
        x, y = 130.0, 95.0
        for k in range(n):
            if k % 11 != 5:  # (else a line of no length)
                x, y = np.clip((x + rng.normal(0, 14), y + rng.normal(0, 14)), 2, 185)
            p.line_to(x, y)
        c.draw_path(p.close() if i % 4 == 1 else p, paint)
    check(ctx, c.scene(), f"join {join}")


@pytest.mark.parametrize("bars", [0, 31, 150])
def test_quads_that_end_above_their_first_row(ctx, bars):
    """Quads over more than 8,192 rows, whose forward differences wrap as the
    reference's do: their first pieces run upward, so that the first row holds
    edges that have ended before it.  They take that row's step and then go on;
    rows are taken several at a time only after that.  With bars beside them the
    lists are of 64 and of 302 edges."""
    rng = np.random.default_rng(4)
    n = 40
    c = Canvas(10 * n + 4 * bars, 300)
    for i in range(n):
        x = 10 * i + rng.uniform(-60, 60, 4)
        top = -float(np.floor(rng.uniform(300, 600)))
        y = np.sort(rng.uniform(7700, 8100, 2))
        p = Path().move_to(x[0], top).quad_to(x[1], y[0], x[2], y[1]).line_to(x[3], top).close()
        for k in range(bars):
            p.add_rect(10 * n + 60 + 4 * k, top, 10 * n + 62.5 + 4 * k, 8000)
        p.fill_type = abi.FILL_EVEN_ODD
        c.draw_path(p, Paint((0.1 + 0.02 * i, 0.9 - 0.02 * i, 0.4, 1.0)))
    check(ctx, c.scene(), "tall quads")
