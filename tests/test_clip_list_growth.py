"""Frames with more lines and pieces across the canvas's borders than the clip
list has room for to begin with (a quarter of 65536 sources and more): exact
sizing grows it and runs the edges again, predicted sizing falls back, and a
graph replay takes the grown size.  Tolerance 0 against the oracle."""
import numpy as np
import pytest

import checkers
from blend2d_amd import scene as S

pytestmark = pytest.mark.gpu

W, H = 96, 64


@pytest.fixture
def amd():
    import blend2d_amd
    if blend2d_amd.lib().bl_amd_device_count() < 1:
        pytest.skip("no HIP device")
    yield blend2d_amd
    blend2d_amd.set_sizing(blend2d_amd.SIZING_EXACT)
    blend2d_amd.set_graph_replay(False)


def _scene(kind, sources, crossing=True):
    """Zigzags whose every source crosses a border (or none does)."""
    rng = np.random.default_rng(sources)
    sc = S.Scene(W, H, S.FMT_A8, 0)
    sc.set_comp_op(S.COMP_OP_PLUS)
    sc.set_fill_style_rgba32(0x02FFFFFF)   # 80 of them stay below 255
    per = 1000
    for k in range(sources // per):
        inside = rng.random((per, 2)) * [W, H]
        if crossing:
            out = rng.random((per, 2)) * [3 * W, 3 * H] - [W, H]
            away = (out > 0).all(axis=1) & (out < [W, H]).all(axis=1)
            out[away] -= [W, 0]
            inside[1::2] = out[1::2]
        sc.set_fill_rule(k & 1)
        if kind == "line":
            sc.fill_polygon([tuple(p) for p in inside])
        else:
            # the point between two neighbours, off to the side
            mid = (inside + np.roll(inside, -1, axis=0)) / 2 + rng.random((per, 2)) * 8 - 4
            mid = np.clip(mid, [-W, -H], [2 * W, 2 * H]) if crossing else np.clip(mid, 0.5, [W - 0.5, H - 0.5])
            pts = np.empty((2 * per + 2, 2))
            pts[0:-2:2], pts[1:-2:2], pts[-2:] = inside, mid, inside[0]
            sc.fill_path([S.CMD_MOVE] + [S.CMD_QUAD, S.CMD_ON] * per + [S.CMD_CLOSE], pts)
    return sc


def _flush(amd, ctx, img, sc):
    img.fill_raw(0)
    ctx.end()
    ctx.begin(img)
    assert amd.replay_into(ctx, sc, []) == []
    ctx.flush()
    return img.download(), ctx.last_stats()


def _target(amd):
    img = amd.BLImage(W, H, S.FMT_A8)
    return img, amd.BLContext(img)


@pytest.mark.parametrize("kind", ["line", "quad"])
def test_exact_sizing_grows_the_list(amd, kind):
    sc = _scene(kind, 80000)
    want, _ = checkers.render_oracle(sc)
    img, ctx = _target(amd)
    got, st = _flush(amd, ctx, img, sc)
    assert st["syncs"] > 3          # edges, counts and end take three
    assert np.array_equal(got, want)
    got, st = _flush(amd, ctx, img, sc)
    assert st["syncs"] == 3         # the list was kept
    assert np.array_equal(got, want)
    ctx.end()


@pytest.mark.parametrize("kind", ["line", "quad"])
def test_predicted_sizing_falls_back(amd, kind):
    sc = _scene(kind, 80000)
    want, _ = checkers.render_oracle(sc)
    img, ctx = _target(amd)
    # an exact frame with segments and bins enough and nothing across a border
    # leaves a list of 64 000
    _, st0 = _flush(amd, ctx, img, _scene("line", 200000, crossing=False))
    amd.set_sizing(amd.SIZING_HISTORY)
    got, st = _flush(amd, ctx, img, sc)
    assert st["fallback"] == 1
    assert st["segments"] < 1.25 * st0["segments"] and st["binned"] < 1.25 * st0["binned"]
    assert np.array_equal(got, want)
    got, st = _flush(amd, ctx, img, sc)
    assert st["fallback"] == 0
    assert np.array_equal(got, want)
    ctx.end()


@pytest.mark.parametrize("kind", ["line", "quad"])
def test_graph_replays_take_the_grown_list(amd, kind):
    sc = _scene(kind, 80000)
    want, _ = checkers.render_oracle(sc)
    img, ctx = _target(amd)
    amd.set_graph_replay(True)
    got, _ = _flush(amd, ctx, img, sc)
    assert np.array_equal(got, want)
    for _ in range(4):
        img.fill_raw(0)
        ctx.replay()
        assert ctx.last_stats()["graph"] == 1
        assert np.array_equal(img.download(), want)
    ctx.end()
