"""Per-image keypoint ranges of a batch where the candidates' capacity takes the
offsets' scan in tiles: images without candidates first, between and last, all images
empty, more candidates than one tile of 4096, against each image alone."""
import numpy as np
import pytest

import imgen
import sift_hip

pytestmark = pytest.mark.gpu

ARGS = (1.6, 3, 3, 0.5, 0.001, 1e6)


def _images(kind):
    flat = np.full((60, 80), 90, np.uint8)
    some = [imgen.generic_image(w, h, seed=w + h, n_blobs=w * h // 150, n_rects=w * h // 900)
            for w, h in ((333, 221), (80, 60), (640, 480), (97, 61))]
    big = imgen.generic_image(1920, 1080, seed=5, n_blobs=14000, n_rects=2300)
    return {"mixed": [flat, some[0], flat, flat, some[1], some[2], some[3], flat],
            "empty": [flat, flat, flat],
            "tiles": [some[0], big, flat, some[2]]}[kind]


@pytest.mark.parametrize("kind", ["mixed", "empty", "tiles"])
@pytest.mark.parametrize("cap", [4096, 66000, 140000])
def test_ranges_of_a_batch(kind, cap, monkeypatch):
    imgs = _images(kind)
    s = sift_hip.Sift(*ARGS)
    alone = [s.detect_and_compute(im) for im in imgs]
    monkeypatch.setenv("SIFT_HIP_CAP_MIN", str(cap))
    monkeypatch.setattr(sift_hip._Ctx, "_ctx", {})  # a context whose capacity starts here
    got = [(k.tobytes(), d.tobytes()) for k, d in sift_hip.Sift(*ARGS).detect_batch(imgs)]
    for h in sift_hip._Ctx._ctx.values():
        sift_hip.free_context(h)
    assert got == [(k.tobytes(), d.tobytes()) for k, d in alone]
    if kind == "tiles":
        assert sum(len(k) for k, _ in alone) > 4096
