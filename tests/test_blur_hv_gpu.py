"""The blur whose two passes share a kernel: levels equal the oracle's bit for
bit. sift_hip_pyramid without the DoG takes it for kernels of 5 to 33 taps; sizes
lie around its tiles (256 x 64 and 64 x 16) and its word-wise edges."""
import ctypes

import numpy as np
import pytest

import devmem
import imgen
import oracle
import sift_hip

pytestmark = pytest.mark.gpu


def _levels(img, params):
    """The Gaussian levels alone (no DoG asked for), octave by octave."""
    sift = sift_hip.Sift(*params)
    h, w = img.shape
    shapes = [(w >> o, h >> o) for o in range(sift.num_octaves)]
    n = sift.num_intervals + 3
    out = np.zeros(sum(n * x * y for x, y in shapes), np.uint8)
    ctx, p = ctypes.c_void_p(), sift.params()
    assert sift_hip.lib().sift_hip_create(ctypes.byref(p), 0, ctypes.byref(ctx)) == 0
    a, s = sift_hip._image_struct(img)
    rc = sift_hip.lib().sift_hip_pyramid(ctx, ctypes.byref(s),
                                         out.ctypes.data_as(ctypes.POINTER(ctypes.c_uint8)), None)
    sift_hip.lib().sift_hip_destroy(ctx)
    assert rc == 0, sift_hip.last_error()
    at, levels = 0, []
    for x, y in shapes:
        levels.append(out[at:at + n * x * y].reshape(n, y, x))
        at += n * x * y
    return levels


# sigma and intervals give the tap counts 5 to 33 (and beyond: the two-pass forms)
@pytest.mark.parametrize("sigma,intervals", [(1.6, 3), (1.6, 5), (2.0, 2), (1.4, 4), (0.9, 3)])
@pytest.mark.parametrize("w,h", [(1, 1), (3, 70), (5, 5), (63, 15), (64, 16), (65, 17), (130, 33),
                                 (255, 63), (256, 64), (257, 129), (333, 221)])
def test_small_tiles_match_the_oracle(w, h, sigma, intervals):
    octaves = max(1, min(3, min(w, h).bit_length() - 1))
    img = imgen.generic_image(w, h, seed=w + h) if min(w, h) > 8 else \
        np.random.default_rng(w * h).integers(0, 256, (h, w), dtype=np.uint8)
    ref = oracle.build_pyramid(oracle.params(sigma, octaves, intervals, 0.5, 0.04, 10.0), img)[0]
    got = _levels(img, (sigma, octaves, intervals, 0.5, 0.04, 10.0))
    for o in range(octaves):
        assert np.array_equal(got[o], ref[o]), o


# one image of over 6 Mpixel takes the large tiles
@pytest.mark.parametrize("w,h,sigma,intervals", [(3001, 2003, 1.6, 3), (2562, 2345, 2.2, 2)])
def test_large_tiles_match_the_oracle(w, h, sigma, intervals):
    img = imgen.generic_image(w, h, seed=5, n_blobs=300, n_rects=200)
    img[:3], img[-3:], img[:, :5], img[:, -2:] = 255, 0, 0, 255
    ref = oracle.build_pyramid(oracle.params(sigma, 2, intervals, 0.5, 0.04, 10.0), img)[0]
    got = _levels(img, (sigma, 2, intervals, 0.5, 0.04, 10.0))
    for o in range(2):
        assert np.array_equal(got[o], ref[o]), o


@pytest.mark.parametrize("pad", [0, 1, 2, 4])
def test_device_frames_of_any_alignment(pad):
    """Rows that are not 4-byte aligned take the two-pass forms: the same result."""
    sift = sift_hip.Sift(1.6, 3, 3, 0.5, 0.04, 10.0)
    img = imgen.generic_image(322, 203, seed=9)
    want_k, want_d = sift.detect_and_compute(img)
    buf, item = devmem.upload_image(img, stride=322 + pad)
    (n,), kp, de, _ = sift.detect_batch_device([item])
    assert n == len(want_k)
    assert devmem.download(kp, n * want_k.itemsize).tobytes() == want_k.tobytes()
    assert devmem.download(de, n * 512).tobytes() == want_d.tobytes()
    buf.free()
