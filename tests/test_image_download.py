"""Image read-back through the pinned chunks: sizes around a chunk (1 MB of
device rows), padded and unpadded rows, caller strides wider than a row,
refused strides, and several threads at once."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import blend2d_amd
    if blend2d_amd.lib().bl_amd_device_count() < 1:
        pytest.skip("no HIP device")
    return blend2d_amd


def _image(amd, w, h, fmt, seed):
    rng = np.random.default_rng(seed)
    px = (rng.integers(0, 256, size=(h, w), dtype=np.uint8) if fmt == amd.FORMAT_A8
          else rng.integers(0, 1 << 32, size=(h, w), dtype=np.uint32))
    img = amd.BLImage(w, h, fmt)
    img.upload(px)
    return img, px


# 1023 and 1024 PRGB32 pixels: 4096-byte device rows, 256 of them a chunk
@pytest.mark.parametrize("w,h", [(1, 1), (3, 5), (1023, 255), (1024, 256), (1023, 257), (1024, 512), (517, 2100), (65535, 9)])
@pytest.mark.parametrize("fmt", [1, 3])
def test_pixels_come_back(amd, w, h, fmt):
    img, px = _image(amd, w, h, fmt, w + h)
    assert np.array_equal(img.download(), px)
    wide = np.full((h, w + 7), 0xA5, dtype=px.dtype)
    r = amd.lib().bl_amd_image_download(img.handle, wide.ctypes.data_as(ctypes.c_void_p), wide.strides[0])
    assert r == 0 and np.array_equal(wide[:, :w], px) and (wide[:, w:] == 0xA5).all()


def test_refused_strides(amd):
    img, px = _image(amd, 10, 4, 1, 1)
    out = np.zeros((4, 10), dtype=np.uint32)
    for stride in (39, 0, -40):
        assert amd.lib().bl_amd_image_download(img.handle, out.ctypes.data_as(ctypes.c_void_p), stride) != 0
    assert not out.any()


def test_threads(amd):
    images = [_image(amd, 700 + 31 * k, 600, 1, k) for k in range(4)]
    bad = []

    def work(img, px):
        for _ in range(8):
            if not np.array_equal(img.download(), px):
                bad.append(1)

    threads = [threading.Thread(target=work, args=a) for a in images]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
