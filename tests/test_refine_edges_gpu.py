"""Refinement next to the image's edges, where the word that holds a row's three
texels reaches past the last column (into the row's padding, the next row or, at
widths that fill the row, past the level): refined keypoints against the oracle's,
bit for bit, with a border of one pixel."""
import numpy as np
import pytest

import oracle
import sift_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w", [61, 62, 63, 64, 128, 129])
@pytest.mark.parametrize("h", [24, 65])
def test_refined_keypoints_at_the_edges(w, h):
    rng = np.random.default_rng(w * 100 + h)
    img = np.kron(rng.integers(0, 256, ((h + 2) // 3, (w + 2) // 3)), np.ones((3, 3)))[:h, :w].astype(np.uint8)
    args = (1.6, 1, 3, 0.5, 0.003, 100.0)
    s, p = sift_hip.Sift(*args), oracle.params(*args)
    s.image_border_width = p.image_border_width = 1
    cand, ref, _, _ = s.detect_stages(img)
    _, _, ocand, oref, _ = oracle.detect_and_compute(p, img, stages=True)
    assert len(ocand) > 0 and cand.tobytes() == ocand.tobytes()
    assert len(ref) == len(oref)
    for f in ("x", "y", "response", "octave", "layer"):
        assert np.array_equal(ref[f], oref[f]), f
