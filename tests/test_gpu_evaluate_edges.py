"""The evaluation kernels at their edges: the 8-bit error over value counts that are no multiple of
four and buffers that wide accesses do not fit (integers: equal), and the image metrics around the
edges of their 32x32-pixel tiles against the float64 loss. The loss is a mean
of FP32 values of size one whose windows cancel at about 1e-7 / C2 (C2 = 9e-4): 1e-5 as elsewhere."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(1, 1), (3, 1), (5, 7), (1021, 3), (1332, 877)])
@pytest.mark.parametrize("shift", [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 3), (3, 2, 1), None])
def test_quantised_error(gsn, context, width, height, shift):
    """`shift`: elements that image, target and result lie past an aligned address; None: no result."""
    rng = np.random.default_rng(width)
    values = width * height * 3
    image = rng.uniform(-0.2, 1.2, values).astype(np.float32)
    target = rng.integers(0, 256, values, dtype=np.uint8)
    i, t, q = shift or (0, 0, 0)
    images = gsn.DeviceBuffer.from_numpy(np.concatenate([np.zeros(i, np.float32), image]))
    targets = gsn.DeviceBuffer.from_numpy(np.concatenate([np.zeros(t, np.uint8), target]))
    results = gsn.DeviceBuffer.from_numpy(np.full(q + values + 5, 77, np.uint8))
    out = (ctypes.c_double * 2)()
    at = lambda buffer, bytes_: ctypes.c_void_p(buffer.ptr.value + bytes_)
    gsn.call("gsn_image_quantized_error", context.handle, width, height, at(images, 4 * i), at(targets, t),
             at(results, q) if shift else None, out)
    expected = np.rint(np.clip(image, 0.0, 1.0) * np.float32(255.0)).astype(np.int64)
    assert out[0] == ((expected - target) ** 2).sum()
    if shift:
        got = results.numpy()
        np.testing.assert_array_equal(got[q:q + values], expected)
        assert (got[:q] == 77).all() and (got[q + values:] == 77).all()


@pytest.mark.parametrize("width,height", [(1, 1), (11, 1), (1, 12), (31, 33), (32, 32), (33, 31), (64, 33), (65, 32),
                                          (97, 5), (5, 130), (257, 191)])
def test_image_metrics(gsn, context, oracle, width, height):
    rng = np.random.default_rng(width * 1000 + height)
    image = rng.uniform(-0.1, 1.1, (height, width, 3)).astype(np.float32)
    target = rng.integers(0, 256, (height, width, 3), dtype=np.uint8)
    metrics = gsn.image_metrics(context, width, height, gsn.DeviceBuffer.from_numpy(image),
                                gsn.DeviceBuffer.from_numpy(target))
    assert abs(metrics["loss"] - oracle.loss_f64(image.astype(np.float64), target)) < 1e-5
    mse = np.mean((np.clip(image, 0, 1).astype(np.float64) - target / 255.0) ** 2)
    assert abs(metrics["mse"] - mse) < 1e-6
