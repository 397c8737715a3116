"""Descriptor windows wider than k_descriptor's (R > 31): the grid of bilinear values
(R <= 47) and the direct form beyond it match the oracle, with keypoints at image
edges and with windows across powers of two (where a sample's neighbour is not a
grid point)."""
import numpy as np
import pytest

import imgen
import oracle
import sift_hip
from parity import DESC_L2_MARGIN, MIN_PR, match_keypoints

pytestmark = pytest.mark.gpu


# R up to ceil(12 sqrt(1/2) sigma 2^(1 + 0.5 / S)): 41 and 39 (grid), 64 and 49 (beyond it)
@pytest.mark.parametrize("sigma,intervals", [(2.0, 2), (2.0, 3), (2.6, 1), (2.6, 4)])
@pytest.mark.parametrize("w,h", [(300, 270), (97, 140), (1100, 90)])
def test_wide_windows_match_the_oracle(w, h, sigma, intervals):
    args = (sigma, 3, intervals, 0.5, 0.03, 10.0)
    img = imgen.generic_image(w, h, seed=w + h, n_blobs=w * h // 300, n_rects=w * h // 900)
    kps, desc = sift_hip.Sift(*args).detect_and_compute(img)
    okps, odesc = oracle.detect_and_compute(oracle.params(*args), img)
    so = okps["size"] / np.exp2(okps["octave"])
    assert (np.ceil(6 * np.sqrt(2) * so) > 31).any()
    m = match_keypoints(okps, kps, odesc, desc)
    assert m["precision"] >= MIN_PR and m["recall"] >= MIN_PR
    assert m["desc_l2_max"] <= DESC_L2_MARGIN, m
