"""GPU parity of forms that only large or unusual frames take: the count pass of
strokes, the count pass of the widest walks, and the widest walk on the widest
row.  Whole-number arithmetic throughout: the tolerance is none."""
import numpy as np
import pytest

from oracle import oracle_py as O
from skity_amd import abi, device
from skity_amd.canvas import Canvas, Paint, Path

from helpers import diff_report

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = device.Context(0)
    yield c
    c.close()


def draw(ctx, sc, **kw):
    surf = device.Surface(ctx, sc.width, sc.height)
    try:
        surf.draw(sc.scene, **kw)
        return surf.read(), surf.stats(), surf.stage_times()
    finally:
        surf.close()


def stroked(i, rng):
    paint = Paint((*rng.uniform(0, 1, 3), 0.7))
    paint.set_style(abi.STYLE_STROKE).set_stroke_width(float(rng.uniform(0.4, 6)))
    return paint.set_stroke_join(i % 3).set_stroke_cap(i // 3 % 3)


def some_strokes(more):
    """Strokes of lines (alone, in runs of a wave's 64 and a chunk's 128 calls,
    some of no length), of curves and of both; and where asked for, 1,024
    polylines above the canvas that take the frame over 1,048,576 segments."""
    rng = np.random.default_rng(7)
    c = Canvas(260, 190)
    for i, n in enumerate((1, 2, 7, 8, 9, 63, 64, 65, 66, 127, 128, 129, 130, 300, 20, 21, 22, 23)):
        p = Path().move_to(130, 95)
        x, y = 130.0, 95.0
        for k in range(n):
            if k % 11 != 5:  # (else a line of no length)
                x, y = np.clip((x + rng.normal(0, 14), y + rng.normal(0, 14)), 2, 185)
            if i > 8 and k % 40 == 17:
                p.quad_to(y, x, x, y)
            elif i > 12 and k % 9 == 3:
                p.cubic_to(y, x, 190 - y, x + 3, x, y)
            elif i > 12 and k % 9 == 6:
                p.conic_to(y, 180 - x, x, y, 0.4 + 0.1 * (k % 12))
            else:
                p.line_to(x, y)
        c.draw_path(p.close() if i % 4 == 1 else p, stroked(i, rng))
    for i in range(1024 if more else 0):
        p = Path().move_to(0, -50)
        for k in range(1024):
            p.line_to(3.0 * (k % 50), -50.0 - (k % 7))
        c.draw_path(p, stroked(i, rng))
    return c.scene()


def test_strokes_counted_before_they_are_written(ctx):
    """The exact form counts the outlines of a frame of more than 1,048,576
    segments; the polylines above the canvas draw nothing."""
    sc = some_strokes(True)
    got, _, stages = draw(ctx, sc)
    assert stages["stroke"][1] == 2  # a count and a write
    seen = some_strokes(False)
    assert diff_report(got, O.render(seen.scene, seen.width, seen.height)) == (0, 0)
    one, _, stages = draw(ctx, seen)
    assert stages["stroke"][1] == 1
    assert np.array_equal(one, got)


def comb(w, teeth, pitch, fill):
    """A closed comb: its rows cross about 2 * teeth edges."""
    c = Canvas(w, 200)
    p = Path().move_to(0.5, 190.25)
    for i in range(teeth):
        x = 2.3 + i * pitch
        p.line_to(x, 10.6 + (i % 7))
        p.line_to(x + 0.5 * pitch, 190.25 - (i % 5))
    p.line_to(w - 0.75, 190.25).close()
    p.fill_type = fill
    c.draw_path(p, Paint((0.2, 0.5, 0.9, 0.9)))
    for k in range(6):  # narrow paths in the same frame
        c.draw_path(Path().add_circle(40 + 150 * k, 100, 30 + 3 * k),
                    Paint((0.9, 0.3 + 0.1 * k, 0.1, 0.6)))
    return c.scene()


@pytest.mark.parametrize("fill", [abi.FILL_WINDING, abi.FILL_EVEN_ODD])
@pytest.mark.parametrize("teeth", [700, 1500])
def test_wide_lists_counted(ctx, teeth, fill):
    """The 32- and 64-slot walks count their planes in a frame whose caller
    sets the bands."""
    sc = comb(int(2.6 * teeth) + 24, teeth, 2.6, fill)
    got, st, stages = draw(ctx, sc, band_rows=32)
    assert stages["walk_count"][1] > 0
    assert st["max_active"] > (1024 if teeth == 700 else 2048)
    assert diff_report(got, O.render(sc.scene, sc.width, sc.height)) == (0, 0)


@pytest.mark.parametrize("band_rows", [0, 32])
@pytest.mark.parametrize("teeth", [1100, 2040])
def test_widest_list_on_the_widest_row(ctx, teeth, band_rows):
    """A 64-slot walk of 16,384 pixel rows takes all but 1.7 KB of a compute
    unit's LDS; its blit scratch lies in the permutation scratch."""
    sc = comb(16384, teeth, 16370.0 / teeth, abi.FILL_WINDING)
    got, st, _ = draw(ctx, sc, band_rows=band_rows)
    assert st["max_active"] > 2048
    assert diff_report(got, O.render(sc.scene, sc.width, sc.height)) == (0, 0)
