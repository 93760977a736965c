"""Curves whose control points are so far away that points overflow while they
are cut or halved.  tests/native/edges_check.cpp compiles the device edge
builder for the host and compares every way a piece can take with the general
builder; two mistakes planted in a copy -- pieces that aren't finite taken as
inside the canvas, and no budget for those that never get flat -- must make it fail or run out of
time.  The reference subdivides such a piece to its recursion limit, which takes
hours, so those that give up have no reference pixels: the fill fails with
BL_ERROR_OUT_OF_MEMORY and the others are drawn."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import checkers
from blend2d_amd import scene as S

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "blend2d_amd", "csrc")
OUT_OF_MEMORY = 0x10000


def _check(tmp_path, n, seed, seconds, edges=None, types=None):
    if not shutil.which("g++"):
        pytest.skip("g++ is missing")
    inc = tmp_path / "blend2d_amd" / "csrc"
    src = tmp_path / "tests" / "native"
    inc.mkdir(parents=True)
    src.mkdir(parents=True)
    for name, text in (("edge_device.h", edges), ("device_types.h", types)):
        (inc / name).write_text(text if text is not None else open(os.path.join(CSRC, name)).read())
    shutil.copy(os.path.join(ROOT, "tests", "native", "edges_check.cpp"), src / "check.cpp")
    exe = tmp_path / "check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-o", str(exe), str(src / "check.cpp")], check=True)
    return subprocess.run([str(exe), str(n), str(seed), str(seconds)], capture_output=True, text=True)


@pytest.mark.parametrize("seed", [1, 2])
def test_every_way_ends_and_agrees(tmp_path, seed):
    res = _check(tmp_path, 60000, seed, 60)
    assert res.returncode == 0, res.stdout + res.stderr


def test_pieces_that_are_not_finite_taken_as_inside_are_caught(tmp_path):
    text = open(os.path.join(CSRC, "edge_device.h")).read()
    planted = text.replace("if (!isfinite(sum)) return kPieceClip;", "").replace("bend > limit)", "!(bend <= limit))")
    assert planted.count("isfinite(sum)") == 0 and planted.count("!(bend <= limit))") == 1
    assert _check(tmp_path, 1, 1, 10, edges=planted).returncode != 0


def test_a_missing_budget_is_caught(tmp_path):
    text = open(os.path.join(CSRC, "device_types.h")).read()
    planted = text.replace("kMaxItemOdd = 1u << 16", "kMaxItemOdd = 0xFFFFFFFFu")
    assert planted != text
    assert _check(tmp_path, 60000, 1, 2, types=planted).returncode != 0


def _path(sc, pts):
    kinds = {3: [S.CMD_MOVE, S.CMD_QUAD, S.CMD_ON], 4: [S.CMD_MOVE, S.CMD_CUBIC, S.CMD_CUBIC, S.CMD_ON]}[len(pts)]
    sc.fill_path(kinds + [S.CMD_CLOSE], np.array(list(pts) + [pts[0]]))


# The first has a piece from inside the canvas to nowhere, which ends; the
# others hold nodes that never get flat (both by edges_check on a 400 x 300
# canvas).
ENDS = [(100.0, 100.0), (4.7e305, 20.0), (200.0, 120.0)]
GIVE_UP = [
    [(232.27141305225439, -2.7357411483562776e+305), (312.8330003192973, 300.0), (248.42205531046613, -3.840695024732771e+304),
     (351.4483914539033, 2.8875984679452043e+305)],
    [(400.00390625, 150.0), (-383.29832064183358, -4.688575486266542e+305), (200.0, -191.36456410147741),
     (-5.8502765299003376e+305, -9.9240836590355797e+304)],
    [(400.00390625, 103.10774132526265), (0.0, -5.5804046675166271e+305), (0.00390625, -2.087054246006666e+305)],
]


@pytest.mark.gpu
def test_far_curves_end_and_the_rest_is_drawn():
    import blend2d_amd as amd
    if amd.lib().bl_amd_device_count() < 1:
        pytest.skip("no HIP device")

    def render(far):
        sc = S.Scene(400, 300, S.FMT_PRGB32, 0xFF102030)
        for k in range(4):
            sc.set_fill_style_rgba32(0xC0FF8040 + 0x10 * k)
            _path(sc, [(20.0 + 90 * k, 30.0), (450.0, 120.0 + 60 * k), (100.0, 260.0)])
            if k < len(far):
                _path(sc, far[k])
        img = amd.BLImage(sc.width, sc.height, sc.format)
        img.fill_raw(sc.clear_value)
        ctx = amd.BLContext(img)
        assert amd.replay_into(ctx, sc, []) == []
        ctx.flush()
        err = ctx.deferred_error()
        got = img.download()
        ctx.end()
        return sc, got, err

    _, _, err = render([ENDS])
    assert err is None
    _, got, err = render(GIVE_UP)
    assert err == (1, OUT_OF_MEMORY)
    plain, same, err = render([])
    want, _ = checkers.render_oracle(plain)
    assert err is None and np.array_equal(same, want)
    assert np.array_equal(got, want)
