"""The largest batches that fit the fixed scratch of the no-allocation entry point are
accepted, and one more row of each frame is refused, with a message. The heights are
those that 256 MiB has held since a step's launch records are counted as 15 of 256
bytes; each call has a context of its own, as the weight tables that a context has
gathered lie in the scratch too."""
import ctypes

import numpy as np
import pytest

import devmem
import sift_hip

pytestmark = pytest.mark.gpu


def _call(sift, buf, w, h, n, out):
    ctx = sift_hip.new_context()
    images = (sift_hip.SiftImage * n)(*[sift_hip.SiftImage(buf.addr, w, h, w)] * n)
    params = (sift_hip.SiftParams * n)(*[sift.params()] * n)
    counts = (ctypes.c_size_t * n)()
    rc = sift_hip.lib().sift_hip_detect_batch_device_noalloc(
        ctx, images, params, n, out[0].addr, out[1].addr, 64, out[2].addr, counts)
    msg = sift_hip.last_error() if rc else ""
    sift_hip.free_context(ctx)
    return rc, msg


@pytest.mark.parametrize("n,w,h,octaves,intervals", [
    (1, 512, 31770, 8, 3), (2, 512, 15938, 8, 3), (2, 640, 15546, 5, 2), (3, 256, 20892, 6, 3)])
def test_largest_batches(n, w, h, octaves, intervals):
    sift = sift_hip.Sift(1.6, octaves, intervals, 0.5, 0.04, 10.0)
    buf = devmem.DeviceBuffer(w * (h + 1))
    buf.upload(np.zeros(buf.nbytes, np.uint8))
    out = [devmem.DeviceBuffer(b) for b in (64 * 28, 64 * 512, 64)]
    rc, msg = _call(sift, buf, w, h, n, out)
    assert rc == 0, msg
    rc, msg = _call(sift, buf, w, h + 1, n, out)
    assert rc == -3 and "scratch" in msg, (rc, msg)
    for b in out + [buf]:
        b.free()
