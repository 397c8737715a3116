"""The fused blur of long kernels on small levels (more than 33 taps): levels equal
the oracle's bit for bit, for levels smaller than the kernel, cut into one or more
tiles of rows, with columns past the image, and with more than 64 KB of LDS."""
import numpy as np
import pytest

import imgen
import oracle
import sift_hip
from test_blur_hv_gpu import _levels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,octaves,sigma,intervals", [
    (640, 480, 5, 1.6, 3), (333, 221, 6, 1.6, 3), (97, 61, 4, 1.6, 5), (700, 41, 4, 2.0, 2),
    (41, 700, 4, 2.0, 2), (64, 257, 3, 1.6, 3), (72, 1030, 3, 1.9, 3), (1920, 1080, 5, 1.6, 3),
    (9, 300, 2, 9.0, 3), (8, 128, 1, 12.0, 1), (3, 5, 2, 30.0, 2), (1, 1, 1, 25.0, 3)])
def test_levels_match_the_oracle(w, h, octaves, sigma, intervals):
    img = imgen.generic_image(w, h, seed=w + 3 * h) if min(w, h) > 8 else \
        np.random.default_rng(w * h).integers(0, 256, (h, w), dtype=np.uint8)
    ref = oracle.build_pyramid(oracle.params(sigma, octaves, intervals, 0.5, 0.04, 10.0), img)[0]
    got = _levels(img, (sigma, octaves, intervals, 0.5, 0.04, 10.0))
    for o in range(octaves):
        assert np.array_equal(got[o], ref[o]), o


def test_batches_on_both_sides_of_the_work_limit():
    """A few frames take the fused form, many the one-pass forms: the same results."""
    sift = sift_hip.Sift(1.6, 5, 3, 0.5, 0.04, 10.0)
    imgs = [imgen.generic_image(480, 270, seed=30 + i) for i in range(24)]
    many = sift.detect_batch(imgs)
    for i in (0, 11, 23):
        k, d = sift.detect_and_compute(imgs[i])
        assert many[i][0].tobytes() == k.tobytes() and many[i][1].tobytes() == d.tobytes()
