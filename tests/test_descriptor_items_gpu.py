"""The descriptor's launches by candidate (many candidates) and by keypoint (few), and
a keypoint's candidate from the list or, past the list's end (more keypoints than the
candidates' capacity), by a search of the offsets: the same keypoints and descriptors,
bit for bit."""
import ctypes

import numpy as np
import pytest

import imgen
import sift_hip

pytestmark = pytest.mark.gpu


def _detect(img, args, cap, monkeypatch):
    """With a context of its own, whose candidate capacity starts at `cap`."""
    monkeypatch.setenv("SIFT_HIP_CAP_MIN", str(cap))
    monkeypatch.setenv("SIFT_HIP_CAP_DIVISOR", "100000000")
    L = sift_hip.lib()
    p = sift_hip.SiftParams()
    L.sift_params_new(ctypes.byref(p), *args)
    h = ctypes.c_void_p()
    assert L.sift_hip_create(ctypes.byref(p), 0, ctypes.byref(h)) == 0
    try:
        keep, im = sift_hip._image_struct(img)
        r = sift_hip.SiftResult()
        assert L.sift_hip_detect(h, ctypes.byref(im), ctypes.byref(r)) == 0, sift_hip.last_error()
        return sift_hip._take_result(r)
    finally:
        L.sift_hip_destroy(h)


@pytest.mark.parametrize("queue", ["0", "1"])
@pytest.mark.parametrize("w,h,sigma", [(97, 61, 1.6), (333, 221, 1.6), (641, 479, 1.6), (301, 223, 2.2)])
def test_by_keypoint_equals_by_candidate(w, h, sigma, queue, monkeypatch):
    monkeypatch.setenv("SIFT_HIP_QUEUE", queue)
    # (the contrast is divided by the intervals; the edge test keeps almost everything)
    args = (sigma, 3, 3, 0.5, 0.0, 1e6)
    img = imgen.generic_image(w, h, seed=w, n_blobs=w * h // 150, n_rects=w * h // 900)
    ncand = len(sift_hip.Sift(*args).detect_stages(img)[0])
    by_candidate = _detect(img, args, 200000, monkeypatch)
    n = len(by_candidate[0])
    assert n > 20
    for cap in (65536, 100000, max(ncand, (2 * n + 2) // 3)):  # the last: fewer than n where it can be
        got = _detect(img, args, cap, monkeypatch)
        assert got[0].tobytes() == by_candidate[0].tobytes(), cap
        assert got[1].tobytes() == by_candidate[1].tobytes(), cap
