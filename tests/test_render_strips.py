"""The analytic-tile kernel at the sizes where it changes form: a tile as four,
two or one workgroups (by the frame's tile count), tiles cut by the canvas
edges, more selected commands than one wave holds, and the pattern fetchers'
wide loads, float reductions and far coordinates.  Tolerance 0 against the
oracle, as everywhere."""
import math

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


# 64 x 16 pixel tiles: 1, 4, 72 and 130 (four strips), 510 (two), 792 (one)
@pytest.mark.parametrize("w,h", [(17, 1), (65, 17), (511, 130), (640, 207), (1025, 480), (1100, 700)])
@pytest.mark.parametrize("fmt", [S.FMT_PRGB32, S.FMT_XRGB32, S.FMT_A8])
def test_tile_forms(amd, w, h, fmt):
    _cmp(amd, S.mixed_scene(w + fmt, w, h, 150, fmt))


@pytest.mark.parametrize("ops", [(S.COMP_OP_PLUS, S.COMP_OP_MULTIPLY, S.COMP_OP_SCREEN, S.COMP_OP_SRC_OVER)])
@pytest.mark.parametrize("w,h", [(120, 70), (700, 300)])
def test_operators(amd, ops, w, h):
    _cmp(amd, S.mixed_scene(w, w, h, 150, S.FMT_PRGB32, ops))


def test_long_command_lists(amd):
    # up to 300 commands of one band reach a tile: several 256-entry chunks
    # and groups of selected entries, solid and not
    sc = S.polygons_scene(3, 90, 40, 300)
    other = S.mixed_scene(4, 90, 40, 300)
    sc.images, sc.cmds = other.images, sc.cmds + other.cmds
    _cmp(amd, sc)


# 61 and 64 texels; scales from a texel covering many pixels to thousands of
# texels a pixel (coordinates past 2^22, where the reduction takes the division)
@pytest.mark.parametrize("texels", [1, 2, 61, 64])
@pytest.mark.parametrize("scale", [3.0, 0.4, 1e-3, 1e-5])
def test_affine_patterns(amd, texels, scale):
    rng = np.random.default_rng(texels)
    sc = S.Scene(333, 150, S.FMT_PRGB32, 0xFF406080)
    img = sc.add_image(S.premultiplied_noise(rng, texels, texels))
    for i in range(18):
        a = 0.37 * i
        sc.set_pattern_quality(i & 1)
        m = [math.cos(a) * scale, math.sin(a) * scale, -math.sin(a) * scale, math.cos(a) * scale, 30.0 * i, 7.0 * i]
        sc.set_fill_style_pattern(img, i % 3, m)
        sc.fill_path(*S.ellipse_path(20.0 + 17 * i, 75.0, 60.0, 70.0))
    _cmp(amd, sc)


# image contents with colours above their alpha; source rows that are not a
# multiple of four pixels, offsets that wrap, clamp and mirror inside a quad
@pytest.mark.parametrize("texels", [3, 61, 64])
def test_translated_patterns(amd, texels):
    rng = np.random.default_rng(texels)
    sc = S.Scene(301, 90, S.FMT_PRGB32, 0xFF406080)
    img = sc.add_image(rng.integers(0, 1 << 32, size=(texels, texels), dtype=np.uint32))
    a8 = sc.add_image(rng.integers(0, 256, size=(texels, texels), dtype=np.uint8), S.FMT_A8)
    for i in range(24):
        sc.set_pattern_quality(1)
        off = (0.5 if i & 1 else 0.0)
        sc.set_fill_style_pattern(a8 if i % 5 == 4 else img, i % 3, [1.0, 0.0, 0.0, 1.0, 7.0 * i - 60.0 + off, 3.0 * i - 20.0 + off])
        sc.fill_path(*S.ellipse_path(12.0 * i, 45.0, 70.0, 44.0))
    _cmp(amd, sc)
