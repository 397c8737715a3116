"""Host images of any width and row stride on their way to the device (staged at
the device pitch, long batches in pieces), and u8 results with the pinned pool
on, off and full: the same results as from device-resident frames, bit for bit."""
import ctypes
import time

import numpy as np
import pytest

import devmem
import imgen
import sift_hip
from test_host_pool_gpu import _with_pool_limit

pytestmark = pytest.mark.gpu

SIFT = (1.6, 3, 3, 0.5, 0.04, 10.0)


def _resident(sift, img):
    buf, item = devmem.upload_image(img)
    (n,), kp, de, _ = sift.detect_batch_device([item])
    kps = devmem.download(kp, n * sift_hip.KEYPOINT_DTYPE.itemsize).tobytes()
    desc = devmem.download(de, n * 512).tobytes()
    buf.free()
    return kps, desc


def _strided(sift, imgs, stride_of):
    """detect_batch through the C entry with rows stride_of(w) bytes apart."""
    n = len(imgs)
    ims, outs, keep = (sift_hip.SiftImage * n)(), (sift_hip.SiftResult * n)(), []
    for i, im in enumerate(imgs):
        h, w = im.shape
        a = np.full((h, stride_of(w)), 255, np.uint8)
        a[:, :w] = im
        keep.append(a)
        ims[i] = sift_hip.SiftImage(a.ctypes.data, w, h, a.shape[1])
    ctx = sift_hip._Ctx.get(0)
    rc = sift_hip.lib().sift_hip_detect_batch(ctx, ims, sift._params_array(n, None), n, outs)
    assert rc == 0, sift_hip.last_error()
    return [tuple(a.tobytes() for a in sift_hip._take_result(outs[i])) for i in range(n)]


# widths around the 64-byte pitch; the last two batches go in several pieces of
# 1 MiB (a piece ending inside an image, and exactly at its end: 1024 x 1024)
@pytest.mark.parametrize("shapes", [
    [(61, 50)], [(63, 64), (64, 63), (65, 40)], [(127, 90), (1, 7), (129, 33)],
    [(1023, 767), (1025, 900), (333, 45)], [(1024, 1024), (1024, 1025), (97, 61)]])
@pytest.mark.parametrize("pad", [0, 1, 64])
def test_host_rows_of_any_width_and_stride(shapes, pad):
    imgs = [imgen.generic_image(w, h, seed=40 + i) for i, (w, h) in enumerate(shapes)]
    sift = sift_hip.Sift(*SIFT)
    assert _strided(sift, imgs, lambda w: w + pad) == [_resident(sift, im) for im in imgs]


@pytest.mark.parametrize("fmt", [sift_hip.PIXEL_RGB8, sift_hip.PIXEL_LUMAA8, sift_hip.PIXEL_RGBA8_CANVAS])
def test_colour_rows_of_odd_widths(fmt):
    rng = np.random.default_rng(3)
    ch = sift_hip.PIXEL_BYTES[fmt]
    imgs = []
    for i, (w, h) in enumerate([(61, 47), (213, 101), (641, 479)]):
        base = imgen.generic_image(w, h, seed=70 + i).astype(np.int16)
        noise = rng.integers(-6, 7, (h, w, ch))
        imgs.append(np.clip(base[:, :, None] + noise, 0, 255).astype(np.uint8))
    sift = sift_hip.Sift(*SIFT)
    grey = [sift_hip.to_luma8(im, fmt) for im in imgs]
    want = [_resident(sift, g) for g in grey]
    got = sift.detect_batch(imgs, formats=[fmt] * 3)
    assert [(k.tobytes(), d.tobytes()) for k, d in got] == want
    served = {}
    with sift_hip.SiftServer(sift, hbm_budget_bytes=2 << 30) as srv:
        for i, im in enumerate(imgs):
            srv.submit(im, i, fmt=fmt)
        end = time.time() + 60
        while len(served) < 3 and time.time() < end:
            for tag, status, k, d, *_ in srv.poll():
                assert status == 0
                served[tag] = (k.tobytes(), d.tobytes())
    assert [served[i] for i in range(3)] == want


def test_u8_results_pooled_plain_and_mixed():
    imgs = [imgen.generic_image(w, h, seed=80 + i) for i, (w, h) in enumerate([(641, 479), (1280, 720), (40, 40)])]
    sift = sift_hip.Sift(*SIFT)

    def run():
        got = sift.detect_batch_u8(imgs, keypoint_convention=sift_hip.KEYPOINTS_WGPU_V2)
        return [(k.tobytes(), d.tobytes()) for k, d in got]

    pooled = _with_pool_limit(None, run)
    assert len(pooled[1][0]) > 1000 and all(len(d) * 28 == len(k) * 128 for k, d in pooled)
    assert _with_pool_limit(0, run) == pooled
    assert _with_pool_limit(1 << 19, run) == pooled  # the first block fits, the second does not
    r = sift_hip.SiftResultU8()
    sift_hip.lib().sift_result_u8_free(ctypes.byref(r))  # an empty result frees nothing
