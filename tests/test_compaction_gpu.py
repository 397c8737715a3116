"""Candidates of images whose row-slot count lies at the limits of the compaction's
forms (one to eight slots per wave with its own scan, a scan before it), against
the oracle's, in order; keypoint ranges of batches of such images."""
import numpy as np
import pytest

import imgen
import oracle
import sift_hip

pytestmark = pytest.mark.gpu


# one octave and 3 intervals: 3 h slots (limits 2048, 4096, 8192, 16384)
@pytest.mark.parametrize("h", [1, 682, 683, 1365, 1366, 2730, 2731, 5461, 5462])
def test_candidates_at_the_slot_limits(h):
    w = 70
    img = imgen.generic_image(w, h, seed=h, n_blobs=h // 8, n_rects=h // 20) if h > 8 else \
        np.random.default_rng(h).integers(0, 256, (h, w), dtype=np.uint8)
    args = (1.6, 1, 3, 0.5, 0.04, 10.0)
    cand, ref, kps, _ = sift_hip.Sift(*args).detect_stages(img)
    _, _, ocand, oref, _ = oracle.detect_and_compute(oracle.params(*args), img, stages=True)
    assert cand.tobytes() == ocand.tobytes()
    assert len(ref) == len(oref)
    assert h == 1 or len(kps) > 0


@pytest.mark.parametrize("heights", [(682, 1, 300), (2731, 2730), (1366,) * 12])
def test_ranges_of_a_batch(heights):
    sift = sift_hip.Sift(1.6, 1, 3, 0.5, 0.04, 10.0)
    imgs = [imgen.generic_image(70, h, seed=h + i, n_blobs=h // 8, n_rects=h // 20) for i, h in enumerate(heights)]
    got = sift.detect_batch(imgs)
    for im, (k, d) in zip(imgs, got):
        k1, d1 = sift.detect_and_compute(im)
        assert k.tobytes() == k1.tobytes() and d.tobytes() == d1.tobytes()
