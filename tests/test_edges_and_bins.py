"""Edge building and binning at the sizes where they change form: segment
regions, the first growth of the segment buffer, curves on and across every
border of the clip box, several scan workgroups, box-only frames, and both
tile sizes of the binning kernels.  Tolerance 0 against the oracle."""
import numpy as np
import pytest

import checkers
from blend2d_amd import scene as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import blend2d_amd
    if blend2d_amd.lib().bl_amd_device_count() < 1:
        pytest.skip("no HIP device")
    return blend2d_amd


def _cmp(amd, sc):
    got, err = amd.render_scene(sc)
    want, oerr = checkers.render_oracle(sc)
    assert err == oerr
    mx, mean, n = checkers.diff_info(got, want)
    assert mx == 0, f"max diff {mx}, mean {mean}, {n} channels differ"


# 900 polygons make about 6800 source lines (one region), 1500 about 11 000 (sixteen)
@pytest.mark.parametrize("count", [1, 900, 1500])
def test_line_sources(amd, count):
    _cmp(amd, S.polygons_scene(count, 300, 200, count))


# few long curves, and (40) more segments than the buffer starts with
@pytest.mark.parametrize("count", [3, 40])
def test_long_curves(amd, count):
    rng = np.random.default_rng(count)
    sc = S.Scene(1500, 1200, S.FMT_A8, 0)
    for k in range(count):
        pts = rng.random((9, 2)) * np.array([1500.0, 1200.0])
        kinds = [S.CMD_QUAD, S.CMD_ON, S.CMD_CUBIC, S.CMD_CUBIC, S.CMD_ON, S.CMD_CUBIC, S.CMD_CUBIC, S.CMD_ON]
        sc.set_fill_rule(k & 1)
        sc.set_fill_style_rgba32(0x80FFFFFF)
        sc.fill_path([S.CMD_MOVE] + kinds + [S.CMD_CLOSE], np.vstack([pts, pts[:1]]))
    _cmp(amd, sc)


# end and control points on, next to and beyond the borders, and pieces at
# most a 256th wide: what the clip list takes and what it does not
@pytest.mark.parametrize("seed", [1, 2, 3])
@pytest.mark.parametrize("w,h", [(33, 17), (200, 130)])
def test_curves_at_the_borders(amd, seed, w, h):
    rng = np.random.default_rng(seed)
    xs = [0.0, w, -1.0 / 256, 1.0 / 256, w - 1.0 / 256, w + 1.0 / 256, -40.0, w + 60.0, w / 2, w / 3]
    ys = [0.0, h, -1.0 / 256, 1.0 / 256, h - 1.0 / 256, h + 1.0 / 256, -30.0, h + 50.0, h / 2, h / 3]
    sc = S.Scene(w, h, S.FMT_A8, 0)
    sc.set_fill_style_rgba32(0x40FFFFFF)
    for k in range(150):
        n = int(rng.integers(3, 9))
        pts, cmds = [], []
        for _ in range(n):
            kind = int(rng.integers(0, 3))
            cmds += [[S.CMD_ON], [S.CMD_QUAD, S.CMD_ON], [S.CMD_CUBIC, S.CMD_CUBIC, S.CMD_ON]][kind]
            x, y = float(rng.choice(xs)), float(rng.choice(ys))
            for _ in range(kind + 1):
                narrow = rng.random() < 0.3   # the next point on (nearly) the same column
                pts.append((x + float(rng.integers(-1, 2)) / 512 if narrow else float(rng.choice(xs)), float(rng.choice(ys))))
        sc.set_fill_rule(k & 1)
        sc.fill_path([S.CMD_MOVE] + cmds + [S.CMD_CLOSE], np.array([pts[-1]] + pts + [pts[-1]]))
    _cmp(amd, sc)


# 2500 bands and 50 000 (band, command) cells; 20 000 cells of four bands
@pytest.mark.parametrize("w,h,count", [(9, 40000, 20), (60, 64, 5000)])
def test_scans_of_several_workgroups(amd, w, h, count):
    sc = S.polygons_scene(5, w, h, count)
    boxes = S.box_scene(6, w, h, 40)
    sc.images, sc.cmds = boxes.images, sc.cmds + boxes.cmds
    _cmp(amd, sc)


def test_many_segments_in_one_frame(amd):
    # 2.4 million segments: the binning kernels' larger tile; every canvas
    # against the same scene on its own and two against the oracle
    scenes = S.glyph_canvases(9, 130, 200)
    outs, errs = amd.render_scenes_batched(scenes)
    assert not any(errs)
    for k in range(0, 130, 13):
        got, err = amd.render_scene(scenes[k])
        assert err == 0 and np.array_equal(got, outs[k])
    for k in (7, 100):
        want, _ = checkers.render_oracle(scenes[k])
        assert np.array_equal(outs[k], want)


# fewer curves than lanes, each a command of its own, from a few pixels to the
# whole canvas: halves of long ones go to lanes that held another command; and
# more curves than lanes, the last ones long
@pytest.mark.parametrize("count", [1, 2, 7, 8, 9, 33, 150])
@pytest.mark.parametrize("kind", ["quad", "cubic", "mixed"])
def test_few_curves(amd, count, kind):
    rng = np.random.default_rng(count)
    sc = S.Scene(1300, 900, S.FMT_A8, 0)
    for k in range(count):
        size = np.array([1300.0, 900.0]) * (0.01 if k % 3 == 1 else 0.12 if k % 3 == 2 else 1.0) * 0.98
        base = (np.array([1300.0, 900.0]) - size) * (0.02 + 0.96 * rng.random(2))
        pts = base + rng.random((6, 2)) * size
        quad = kind == "quad" or (kind == "mixed" and k & 1)
        sc.set_fill_rule(k & 1)
        sc.set_fill_style_rgba32(0x60FFFFFF)
        if quad:
            sc.fill_path([S.CMD_MOVE, S.CMD_QUAD, S.CMD_ON, S.CMD_QUAD, S.CMD_ON, S.CMD_CLOSE], np.vstack([pts[:5], pts[:1]]))
        else:
            sc.fill_path([S.CMD_MOVE, S.CMD_CUBIC, S.CMD_CUBIC, S.CMD_ON, S.CMD_CLOSE], np.vstack([pts[:4], pts[:1]]))
    _cmp(amd, sc)


# curves of all lengths that leave the canvas, from one to many a wave: parts
# inside it go to the wave's list until that is full, further segments past the
# staging buffer
@pytest.mark.parametrize("count", [1, 5, 70, 600])
@pytest.mark.parametrize("kind", ["quad", "cubic"])
def test_curves_leaving_the_canvas(amd, count, kind):
    rng = np.random.default_rng(count)
    size = np.array([900.0, 700.0])
    sc = S.Scene(900, 700, S.FMT_A8, 0)
    for k in range(count):
        pts = (rng.random((5, 2)) * (3.0 if k % 3 else 1.1) - (1.0 if k % 3 else 0.05)) * size
        sc.set_fill_rule(k & 1)
        sc.set_fill_style_rgba32(0x30FFFFFF)
        if kind == "quad":
            sc.fill_path([S.CMD_MOVE, S.CMD_QUAD, S.CMD_ON, S.CMD_QUAD, S.CMD_ON, S.CMD_CLOSE], pts[[0, 1, 2, 3, 4, 0]])
        else:
            sc.fill_path([S.CMD_MOVE, S.CMD_CUBIC, S.CMD_CUBIC, S.CMD_ON, S.CMD_CLOSE], pts[[0, 1, 2, 3, 0]])
    _cmp(amd, sc)
