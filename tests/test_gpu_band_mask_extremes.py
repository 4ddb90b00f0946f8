"""The rasterisers' band mask at conics far outside what a projection makes (it adds 0.3 to a
covariance's diagonal), which gsn_render_tiles takes all the same: entries down to the smallest and up
to the largest floats, where a reciprocal or a product leaves the range of normal numbers. A band that
holds a pixel with alpha at or above 1/255 (the rasteriser's rule in FP64, at a threshold 0.1% above)
is never dropped."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# Ranges of the two diagonal entries, each log-uniform.
RANGES = [(1e36, 3e38, 1e-3, 1e2), (1e-3, 1e2, 1e36, 3e38), (1e-40, 1e-34, 1e-3, 1e3), (1e-3, 1e3, 1e-40, 1e-34),
          (1e-38, 1e38, 1e-38, 1e38), (1e-25, 1e-18, 1e-25, 1e-18), (1e17, 1e20, 1e17, 1e20)]


@pytest.mark.parametrize("a_low,a_high,c_low,c_high", RANGES)
@pytest.mark.parametrize("correlated", [False, True])
def test_no_band_lost(gsn, context, a_low, a_high, c_low, c_high, correlated):
    rng = np.random.default_rng(17)
    count = 8000
    a = np.exp(rng.uniform(np.log(a_low), np.log(a_high), count))
    c = np.exp(rng.uniform(np.log(c_low), np.log(c_high), count))
    b = rng.uniform(-1, 1, count) * np.sqrt(a) * np.sqrt(c) * correlated
    means = np.round(rng.uniform(-4, 20, (count, 2)) * 2) / 2  # many on a pixel's row or column
    splats = np.stack([means[:, 0], means[:, 1], a, b, c, rng.uniform(1 / 255, 1, count)], axis=1).astype(np.float32)
    device_splats = gsn.DeviceBuffer.from_numpy(splats)
    origins = gsn.DeviceBuffer.from_numpy(np.zeros((count, 2), np.int32))
    masks = gsn.DeviceBuffer((count,), np.int32)
    gsn.call("gsn_selftest_band_mask", context.handle, device_splats.ptr, origins.ptr, count, masks.ptr)
    context.synchronize()
    s = splats.astype(np.float64)[:, :, None, None]
    rows, columns = np.mgrid[:16, :16]
    dx, dy = s[:, 0] - columns, s[:, 1] - rows
    power = -0.5 * (s[:, 2] * dx * dx + s[:, 4] * dy * dy) - s[:, 3] * dx * dy
    alpha = np.minimum(0.99, s[:, 5] * np.exp(np.minimum(power, 0.0)))
    needed = ((power <= 0) & (alpha >= 1.001 / 255)).reshape(count, 4, 64).any(axis=2)
    kept = (masks.numpy()[:, None] >> np.arange(4)) & 1 != 0
    assert needed.any() and not (needed & ~kept).any()
