"""The box compositor at the sizes where it changes form: groups of 256 x 16
pixels cut by the canvas, boxes that start and end inside a quad of pixels or a
wave's four rows, canvases whose first fill replaces the pixels and canvases
whose contents stay, masks and images at every alignment, and more commands
than one wave holds.  Tolerance 0 against the oracle, as everywhere."""
import numpy as np
import pytest

import checkers
from blend2d_amd import scene as S

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (5, 3), (255, 17), (256, 16), (257, 33), (530, 70)]


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


def _boxes(sc, rng, n, fractions):
    for _ in range(n):
        x, y = (int(rng.integers(0, m)) for m in (sc.width, sc.height))
        w, h = (int(rng.integers(1, m + 1)) for m in (sc.width, sc.height))
        f = float(rng.integers(0, 4)) / 4 if fractions else 0.0
        sc.set_fill_style_rgba32(int(rng.integers(0, 1 << 32)))
        sc.fill_rect_d(x + f, y + f, w + f, h)


# the first fill: none (contents stay), opaque, translucent, opaque over a part
@pytest.mark.parametrize("first", ["none", "opaque", "translucent", "part"])
@pytest.mark.parametrize("fmt", [S.FMT_PRGB32, S.FMT_XRGB32, S.FMT_A8])
@pytest.mark.parametrize("w,h", SIZES)
def test_solid_boxes(amd, w, h, fmt, first):
    rng = np.random.default_rng(w + fmt)
    for fractions in (False, True):
        sc = S.Scene(w, h, fmt, 0 if fmt == S.FMT_A8 else 0xFF406080)
        if first == "part":
            sc.set_fill_style_rgba32(0xFF123456)
            sc.fill_rect_d(0.0, 0.0, float(max(1, w - 1)), float(h))
        elif first != "none":
            sc.fill_all_rgba32(0xFF123456 if first == "opaque" else 0x80123456)
        # whole-canvas layers, then boxes: one value per wave, then per pixel
        for _ in range(2):
            sc.set_fill_style_rgba32(int(rng.integers(0, 1 << 32)))
            sc.fill_all()
        _boxes(sc, rng, 90, fractions)     # more than 64 in a band
        _cmp(amd, sc)


@pytest.mark.parametrize("op", [S.COMP_OP_SRC_COPY, S.COMP_OP_PLUS, S.COMP_OP_MULTIPLY, S.COMP_OP_SCREEN])
def test_operators(amd, op):
    rng = np.random.default_rng(op)
    sc = S.Scene(300, 40, S.FMT_PRGB32, 0xFF406080)
    sc.fill_all_rgba32(0xFF123456)
    sc.set_comp_op(op)
    sc.fill_all_rgba32(0x80402010)
    _boxes(sc, rng, 20, False)
    _cmp(amd, sc)


@pytest.mark.parametrize("fmt", [S.FMT_PRGB32, S.FMT_XRGB32, S.FMT_A8])
@pytest.mark.parametrize("w,h", SIZES)
def test_blits(amd, w, h, fmt):
    rng = np.random.default_rng(w)
    sc = S.Scene(w, h, fmt, 0 if fmt == S.FMT_A8 else 0xFF406080)
    imgs = [sc.add_image(rng.integers(0, 1 << 32, size=(h, w), dtype=np.uint32), S.FMT_PRGB32),
            sc.add_image(rng.integers(0, 1 << 32, size=(9, 61), dtype=np.uint32), S.FMT_XRGB32),
            sc.add_image(S.premultiplied_noise(rng, 2, 1)),
            sc.add_image(rng.integers(0, 256, size=(9, 33), dtype=np.uint8), S.FMT_A8)]
    sc.blit_image(S.BLIT_I, imgs[0], (0, 0))
    for i in range(24):
        img = imgs[i % 4]
        x, y = int(rng.integers(-8, w)), int(rng.integers(-8, h))
        sc.set_global_alpha(1.0 if i & 1 else 0.7)
        sc.blit_image(S.BLIT_I, img, (x, y))
        sc.blit_image(S.BLIT_D, img, (x + 0.4, y - 0.7))
        sc.blit_image(S.BLIT_SCALED_I, img, (x, y, int(rng.integers(1, 300)), int(rng.integers(1, 40))))
    _cmp(amd, sc)


@pytest.mark.parametrize("fmt", [S.FMT_PRGB32, S.FMT_A8])
@pytest.mark.parametrize("w,h", SIZES)
def test_masks(amd, w, h, fmt):
    rng = np.random.default_rng(h)
    for gradient in (False, True):
        sc = S.Scene(w, h, fmt, 0 if fmt == S.FMT_A8 else 0xFF406080)
        mask = sc.add_image(rng.integers(0, 256, size=(h + 3, w + 5), dtype=np.uint8), S.FMT_A8)
        for i in range(12):
            sc.set_fill_style_rgba32(int(rng.integers(0, 1 << 32)))
            if gradient and i & 1:
                sc.set_fill_style_gradient(S.GRADIENT_LINEAR, [0.0, 0.0, float(w), float(h)],
                                           [(0.0, 0xC0FF0000), (1.0, 0x800000FF)])
            sc.set_global_alpha(1.0 if i % 3 else 0.6)
            sc.fill_mask(S.MASK_I, mask, (int(rng.integers(-6, w)), int(rng.integers(-6, h))))
        _cmp(amd, sc)


# reflected, repeated and clamped patterns whose neighbouring texels are
# neighbours, the same one, or the two ends of a row
@pytest.mark.parametrize("texels", [1, 2, 3, 64])
@pytest.mark.parametrize("fmt", [S.FMT_PRGB32, S.FMT_XRGB32, S.FMT_A8])
def test_scaled_patterns(amd, texels, fmt):
    rng = np.random.default_rng(texels)
    sc = S.Scene(520, 40, S.FMT_PRGB32, 0xFF406080)
    shape = (texels, texels)
    img = (sc.add_image(rng.integers(0, 256, size=shape, dtype=np.uint8), fmt) if fmt == S.FMT_A8
           else sc.add_image(rng.integers(0, 1 << 32, size=shape, dtype=np.uint32), fmt))
    sc.set_pattern_quality(1)
    for i in range(27):
        m = [(0.3, 1.0, 2.7)[i % 3] * (-1.0 if i & 1 else 1.0), 0.0, 0.0, (0.5, 1.9)[i & 1], 19.3 * i, 3.1 * i]
        sc.set_fill_style_pattern(img, i // 9, m)
        sc.fill_rect_d(float(19 * i), 0.0, 40.0, 40.0)
        sc.set_fill_style_pattern(img, i // 9, [1.0, 0.0, 0.0, 1.0, 7.25 * i, 3.5 * i])
        sc.fill_rect_d(float(19 * i), 0.0, 21.0, 20.0)
    _cmp(amd, sc)
