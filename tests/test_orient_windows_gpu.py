"""Orientations of keypoints whose window sizes lie on both sides of the staging
forms' limits (R = 9 / 10, 12 / 13, 16 / 17: more than 16 is not staged), with many
windows across the image's edges, against the oracle within the contract's
tolerances (0.05 px, 1 degree; 99.5% matched)."""
import numpy as np
import pytest

import imgen
import oracle
import sift_hip
from parity import MIN_PR, match_keypoints

pytestmark = pytest.mark.gpu


# layers 1..3 of the one octave have R = round(4.5 sigma 2^(l/3)) around these
@pytest.mark.parametrize("sigma", [0.7, 1.25, 1.6, 1.9, 2.2, 2.6, 3.0])
@pytest.mark.parametrize("w,h", [(301, 223), (90, 33)])
def test_orientations_by_window_size(sigma, w, h):
    rng = np.random.default_rng(int(sigma * 100) + w)
    img = imgen.generic_image(w, h, seed=int(sigma * 100), n_blobs=w * h // 120, n_rects=w * h // 900)
    img = np.clip(img.astype(np.int32) + rng.integers(-6, 7, img.shape), 0, 255).astype(np.uint8)
    args = (sigma, 1, 3, 0.5, 0.01, 20.0)
    kps, _ = sift_hip.Sift(*args).detect_and_compute(img)
    okps, _ = oracle.detect_and_compute(oracle.params(*args), img)
    m = match_keypoints(okps, kps)
    assert w < 300 or m["n_ref"] > 100
    assert m["precision"] >= MIN_PR and m["recall"] >= MIN_PR
