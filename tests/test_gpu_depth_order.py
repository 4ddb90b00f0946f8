"""The depth order on either side of the 24,576 Gaussians up to which it is made by counting, through the
lists of a one-tile screen: ids by (depth bits, id), equal."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 2, 255, 256, 257, 513, 24_575, 24_576, 24_577])
@pytest.mark.parametrize("distinct", [1, 50, 1 << 30])
def test_depth_order(gsn, context, count, distinct):
    rng = np.random.default_rng(count)
    depths = (1 + rng.integers(0, distinct, count)).astype(np.float32)
    visible = rng.random(count) < 0.8
    visible[0] = True
    rects = np.where(visible[:, None], np.array([[0, 0, 1, 1]]), -9).astype(np.int32)
    records = int(visible.sum())
    camera = gsn.Camera.make(16, 16, 1.0, 1.0, 0.0, 0.0)
    offsets = gsn.DeviceBuffer.from_numpy(np.concatenate([[0], np.cumsum(visible)]).astype(np.int32))
    device_rects, device_depths = gsn.DeviceBuffer.from_numpy(rects), gsn.DeviceBuffer.from_numpy(depths)
    ids, tile_offsets = gsn.DeviceBuffer((records,), np.int32), gsn.DeviceBuffer((2,), np.int64)
    gsn.call("gsn_build_tile_lists", context.handle, ctypes.byref(camera), count, device_rects.ptr, device_depths.ptr,
             offsets.ptr, records, ids.ptr, tile_offsets.ptr, None)
    context.synchronize()
    order = np.argsort(depths, kind="stable")
    np.testing.assert_array_equal(ids.numpy(), order[visible[order]])
