"""Descriptors of narrow and wide windows (R 14 to 31: one to 18 staged words per row,
three to eight bands of grid rows) along images that cross the powers of two, where a
window's f32 rows can skip a texel row, and at their edges: against the oracle."""
import numpy as np
import pytest

import imgen
import oracle
import sift_hip
from parity import DESC_L2_MARGIN, MIN_PR, match_keypoints

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sigma,intervals", [(0.8, 3), (1.0, 5), (1.3, 2), (1.6, 3), (1.69, 6)])
@pytest.mark.parametrize("w,h", [(64, 2200), (2200, 64), (300, 301)])
def test_windows_match_the_oracle(w, h, sigma, intervals):
    args = (sigma, 2, intervals, 0.3, 0.02, 10.0)
    img = imgen.generic_image(w, h, seed=w + h, n_blobs=w * h // 200, n_rects=w * h // 800)
    kps, desc = sift_hip.Sift(*args).detect_and_compute(img)
    okps, odesc = oracle.detect_and_compute(oracle.params(*args), img)
    assert len(okps) > 50
    m = match_keypoints(okps, kps, odesc, desc)
    assert m["precision"] >= MIN_PR and m["recall"] >= MIN_PR
    assert m["desc_l2_max"] <= DESC_L2_MARGIN, m
