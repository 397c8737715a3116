"""Device frames whose rows lie far apart: a frame is described the same, bit for
bit, whatever stride it is given with. Rows 64 MiB apart put a tile's rows more than
4 GiB apart, past what 32-bit offsets from its first row reach; a stride of 2 GiB or
more does not fit an int."""
import numpy as np
import pytest

import devmem
import sift_hip

pytestmark = pytest.mark.gpu


def _blocks(w, h):
    a = np.random.default_rng(3).integers(0, 256, (h // 16 + 2, w // 16 + 2), dtype=np.uint8)
    return np.kron(a, np.ones((16, 16), np.uint8))[:h, :w].copy()


def _upload(img, stride):
    """The rows `stride` bytes apart; what lies between them is left as it is."""
    h, w = img.shape
    buf = devmem.DeviceBuffer((h - 1) * stride + w)
    for y in range(h):
        buf.upload(img[y], offset=y * stride)
    return buf


def _compare(sigma, w, h, stride, least):
    img = _blocks(w, h)
    sift = sift_hip.Sift(sigma, 2, 3, 0.5, 0.0, 1000.0)
    want_k, want_d = sift.detect_and_compute(img)
    assert len(want_k) >= least
    buf = _upload(img, stride)
    (n,), kp, de, _ = sift.detect_batch_device([(buf.addr, w, h, stride)])
    got_k, got_d = devmem.download(kp, n * want_k.itemsize), devmem.download(de, n * 512)
    buf.free()
    assert n == len(want_k)
    assert got_k.tobytes() == want_k.tobytes()
    assert got_d.tobytes() == want_d.tobytes()


# base kernels of 7, 37, 49 and 81 taps: both passes in one kernel up to 33 taps and, on
# small levels, beyond
@pytest.mark.parametrize("sigma", [1.6, 9.0, 12.0, 20.0])
@pytest.mark.parametrize("stride", [64 << 20, (64 << 20) + 1])
def test_rows_far_apart(sigma, stride):
    _compare(sigma, 96, 200, stride, 10)


@pytest.mark.parametrize("sigma", [1.6, 9.0])
@pytest.mark.parametrize("stride", [(2 << 30) + 4, (2 << 30) + 1])
def test_strides_past_an_int(sigma, stride):
    _compare(sigma, 120, 24, stride, 1)


@pytest.mark.parametrize("w", [33, 34, 35, 36, 61])
def test_last_row_ends_the_buffer(w):
    """Rows on word boundaries whose last word is not the frame's alone."""
    _compare(1.6, w, 200, (w + 3) // 4 * 4, 1)
