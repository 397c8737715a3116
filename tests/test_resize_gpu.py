"""The octave step's kernels of both Lanczos3 passes (large tiles from 2.05 Mpixel,
small ones below) on sizes whose halving is exact and on sizes whose windows
shift, at the edges of their tiles: every octave base equals the oracle's."""
import numpy as np
import pytest

import imgen
import oracle
import sift_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,octaves", [
    (2051, 1003, 3), (4101, 501, 2), (70, 30001, 2), (1922, 1090, 2), (15361, 135, 3),  # large tiles
    (2, 2, 2), (3, 2, 2), (5, 7, 2), (33, 35, 3), (128, 8, 3), (129, 9, 3), (130, 130, 3), (259, 61, 4)])
def test_octave_bases_match_the_oracle(w, h, octaves):
    rng = np.random.default_rng(w + h)
    # blocks of black and white (overshoots on both sides of the range) and noise
    img = (rng.integers(0, 2, (h // 9 + 1, w // 11 + 1)) * 255).repeat(9, 0).repeat(11, 1)[:h, :w]
    img = np.where(rng.random((h, w)) < 0.3, rng.integers(0, 256, (h, w)), img).astype(np.uint8)
    # no blur to speak of before the steps: sigma at the assumed blur, long intervals apart
    ref = oracle.build_pyramid(oracle.params(0.5, octaves, 1, 0.5, 0.04, 10.0), img)[0]
    got, _ = sift_hip.Sift(0.5, octaves, 1, 0.5, 0.04, 10.0).pyramid(img)
    for o in range(octaves):
        assert np.array_equal(got[o], ref[o]), o
