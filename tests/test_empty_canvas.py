"""Canvases and bands that no command touches, and batches in which a context
recorded nothing.  A band without commands goes to no kernel: the compositor of
words would read past the end of an A8 canvas.  An empty canvas has no first
command to look at: the command behind the last one is whatever an earlier,
larger frame left there, and its style may lie outside the style table.  On the
CPU both rules are compiled for the host with tables that end at a page without
access (tests/native/group_fresh_check.cpp); without the look at the counts,
taken out of a copy, the check dies or fails."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import checkers
from blend2d_amd import scene as S

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "blend2d_amd", "csrc")


def _check(tmp_path, text=None):
    if not shutil.which("g++"):
        pytest.skip("g++ is missing")
    inc = tmp_path / "blend2d_amd" / "csrc"
    src = tmp_path / "tests" / "native"
    inc.mkdir(parents=True)
    src.mkdir(parents=True)
    for name in ("device_types.h", "raster_device.h", "group_device.h"):
        shutil.copy(os.path.join(CSRC, name), inc / name)
    if text is not None:
        (inc / "group_device.h").write_text(text)
    shutil.copy(os.path.join(ROOT, "tests", "native", "group_fresh_check.cpp"), src / "check.cpp")
    exe = tmp_path / "check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-o", str(exe), str(src / "check.cpp")], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True)


def test_groups_of_an_empty_canvas_read_no_command(tmp_path):
    res = _check(tmp_path)
    assert res.returncode == 0 and "mismatches 0" in res.stdout, res.stderr


@pytest.mark.parametrize("rule", ["if (cv.n_cmds == 0u) return false;", "if (listed == 0u) return kBandEmpty;"])
def test_without_a_look_at_the_counts_the_check_fails(tmp_path, rule):
    text = open(os.path.join(CSRC, "group_device.h")).read()
    planted = text.replace(rule, "")
    assert planted != text
    assert _check(tmp_path, planted).returncode != 0


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [S.FMT_A8, S.FMT_PRGB32])
def test_bands_without_commands_go_to_no_kernel(fmt):
    import blend2d_amd as amd
    if amd.lib().bl_amd_device_count() < 1:
        pytest.skip("no HIP device")
    sc = S.Scene(256, 256, fmt, 0x21)
    sc.set_fill_style_rgba32(0xC0FF8040)
    sc.fill_polygon([(20.0, 40.0), (200.0, 50.0), (90.0, 90.0)])
    img = amd.BLImage(sc.width, sc.height, sc.format)
    img.fill_raw(sc.clear_value)
    ctx = amd.BLContext(img)
    assert amd.replay_into(ctx, sc, []) == []
    ctx.flush()
    assert ctx.last_stats()["render_kernels"] == 1     # the tile kernel alone
    want, _ = checkers.render_oracle(sc)
    assert np.array_equal(img.download(), want)
    ctx.end()


@pytest.mark.gpu
@pytest.mark.parametrize("empty", [(3,), (1,), (0,), (0, 1, 3)])
def test_batches_with_empty_contexts(empty):
    import blend2d_amd as amd
    if amd.lib().bl_amd_device_count() < 1:
        pytest.skip("no HIP device")
    scenes = [S.box_scene(20 + k, 300 - 40 * k, 50, 30) for k in range(4)]
    few = [S.polygons_scene(30 + k, 300 - 40 * k, 50, 5) if k & 1 else S.box_scene(40 + k, 300 - 40 * k, 50, 3) for k in range(4)]
    targets = [amd.BLImage(sc.width, sc.height, sc.format) for sc in scenes]
    ctxs = [amd.BLContext(t) for t in targets]
    batch = amd.BLBatch()
    for ctx in ctxs:
        batch.add(ctx)
    # a batch that fills every context, so that the tables hold its commands
    for frame, skip in ((scenes, ()), (few, empty)):
        for sc, t, ctx, k in zip(frame, targets, ctxs, range(4)):
            t.fill_raw(sc.clear_value)
            ctx.end()
            ctx.begin(t)
            if k in skip:
                continue
            images = []
            for fmt, px in sc.images:
                im = amd.BLImage(px.shape[1], px.shape[0], fmt)
                im.upload(px)
                images.append(im)
            assert amd.replay_into(ctx, sc, images) == []
        batch.flush()
        for k in range(4):
            got = targets[k].download()
            if k in skip:
                assert np.all(got == frame[k].clear_value), k
            else:
                want, err = checkers.render_oracle(frame[k])
                assert err == 0 and np.array_equal(got, want), k
    for ctx in ctxs:
        ctx.end()
