"""The extremum test on strips of 64 columns where a strip ends inside an 8-byte
word, at a word's or a strip's edge or one pixel past it, and on images narrower
than a word: candidates against the oracle's, in order, and (with no border, where
the columns outside the image count) against the row-wise kernel's results."""
import numpy as np
import pytest

import imgen
import oracle
import sift_hip

pytestmark = pytest.mark.gpu

WIDTHS = [12, 15, 16, 17, 63, 64, 65, 71, 72, 73, 127, 128, 129, 135]


def _image(w, h):
    # noise over blobs: extrema in every column, also next to the edges
    img = np.random.default_rng(w * 1000 + h).integers(0, 256, (h, w)).astype(np.float32)
    ker = np.array([1, 4, 6, 4, 1], np.float32) / 16
    for ax in (0, 1):
        img = np.apply_along_axis(lambda r: np.convolve(np.pad(r, 2, mode="edge"), ker, "valid"), ax, img)
    return np.clip((img - 128) * 3 + 128, 0, 255).astype(np.uint8)


@pytest.mark.parametrize("w", WIDTHS)
def test_candidates_at_strip_edges(w):
    img = _image(w, 61)
    args = (1.6, 1, 3, 0.5, 0.001, 100.0)
    cand, ref, _, _ = sift_hip.Sift(*args).detect_stages(img)
    _, _, ocand, oref, _ = oracle.detect_and_compute(oracle.params(*args), img, stages=True)
    assert w < 60 or len(cand) > 0  # at 12 two columns are tested
    assert cand.tobytes() == ocand.tobytes()
    assert len(ref) == len(oref)


@pytest.mark.parametrize("w", [1, 5, 7, 8, 9] + WIDTHS)
def test_no_border_against_the_row_wise_kernel(w):
    img = _image(w, 35)
    a = sift_hip.Sift(1.6, 1, 3, 0.5, 0.0, 100.0)
    b = sift_hip.Sift(1.6, 1, 4, 0.5, 0.0, 100.0)
    a.image_border_width = b.image_border_width = 0
    together = a.detect_batch([img, img], [a, b])  # 3 and 4 intervals: the row-wise kernel
    for p, (k, d) in zip((a, b), together):
        k1, d1 = p.detect_and_compute(img)
        assert k.tobytes() == k1.tobytes() and d.tobytes() == d1.tobytes()
