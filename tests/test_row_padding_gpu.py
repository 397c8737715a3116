"""Images whose width is not a multiple of four: the bytes between a level's
width and its pitch are not part of any result. Frames are described after calls
that leave other bytes there (a black, a white and a textured frame of the same
layout), and every time the same, bit for bit."""
import numpy as np
import pytest

import imgen
import sift_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1025, 900), (1023, 767), (333, 245), (62, 61)])
def test_results_do_not_depend_on_row_padding(w, h):
    sift = sift_hip.Sift(1.6, 3, 3, 0.5, 0.04, 10.0)
    img = imgen.generic_image(w, h, seed=41)
    got = []
    for before in (np.zeros((h, w + 3), np.uint8), np.full((h, w + 3), 255, np.uint8),
                   imgen.generic_image(w + 3, h, seed=42)):
        sift.detect_and_compute(before)
        k, d = sift.detect_and_compute(img)
        got.append((k.tobytes(), d.tobytes()))
    assert got[0] == got[1] == got[2]
