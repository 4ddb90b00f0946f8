"""gsn_build_tile_lists against a NumPy stable sort by (tile, depth, id), over grids and counts on
either side of the edges of its decomposition: 32x32-tile parts, 8x8-tile regions,
64-entry queues, 4,096-entry lists and chunks of 256 to 8,192 entries, all of which count and
write (at least a quarter record per entry and part). Integers: equal."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (tiles_x, tiles_y, count, largest rectangle side in tiles)
CASES = [
    (1, 1, 1, 1), (1, 1, 300, 1), (4, 4, 64, 4), (8, 8, 65, 8), (9, 8, 257, 9), (7, 17, 1025, 5), (33, 32, 4097, 12),
    (64, 40, 5000, 12),
    (120, 68, 3000, 120),  # rectangles up to the whole screen
    (1, 300, 700, 4), (300, 1, 700, 4),  # strips
    (512, 511, 12_000, 9), (513, 130, 40_000, 30),  # many parts, ragged last ones
    (40, 33, 1_500_000, 2),  # chunks of 4,096 entries
    (120, 68, 750_000, 3),  # chunks of 8,192 entries, two lists each
    (65_535, 1, 500, 4), (1, 65_535, 500, 4),  # the largest
]


@pytest.mark.parametrize("tiles_x,tiles_y,count,side", CASES)
def test_tile_lists_equal_a_stable_sort(gsn, context, tiles_x, tiles_y, count, side):
    rng = np.random.default_rng(tiles_x * 1009 + tiles_y * 31 + count)
    width, height = rng.integers(1, min(side, tiles_x) + 1, count), rng.integers(1, min(side, tiles_y) + 1, count)
    x0 = (rng.random(count) ** 2 * (tiles_x - width + 1)).astype(np.int64)  # crowded towards one corner
    y0 = (rng.random(count) ** 2 * (tiles_y - height + 1)).astype(np.int64)
    rects = np.stack([x0, y0, x0 + width, y0 + height], axis=1).astype(np.int32)
    depths = rng.integers(1, 1 + count // 3 + 1, count).astype(np.float32)  # many equal depths
    visible = rng.random(count) < 0.9 if count > 1 else np.ones(1, bool)
    rects[~visible] = -12345  # the projection leaves culled Gaussians' rectangles unwritten
    areas = np.where(visible, width * height, 0)
    record_count = int(areas.sum())

    owner = np.repeat(np.arange(count), areas)
    local = np.arange(record_count) - (np.cumsum(areas) - areas)[owner]
    tile = (y0[owner] + local // width[owner]) * tiles_x + x0[owner] + local % width[owner]
    order = np.lexsort((owner, depths[owner], tile))
    expected_offsets = np.searchsorted(tile[order], np.arange(tiles_x * tiles_y + 1))

    camera = gsn.Camera.make(16 * tiles_x, 16 * tiles_y, 1.0, 1.0, 0.0, 0.0)
    assert (camera.tile_count_x, camera.tile_count_y) == (tiles_x, tiles_y)
    offsets = gsn.DeviceBuffer.from_numpy(np.concatenate([[0], np.cumsum(areas)]).astype(np.int32))
    ids = gsn.DeviceBuffer((max(record_count, 1),), np.int32)
    tile_offsets = gsn.DeviceBuffer((tiles_x * tiles_y + 1,), np.int64)
    keys = gsn.DeviceBuffer((max(record_count, 1),), np.uint64)
    device_rects, device_depths = gsn.DeviceBuffer.from_numpy(rects), gsn.DeviceBuffer.from_numpy(depths)
    gsn.call("gsn_build_tile_lists", context.handle, ctypes.byref(camera), count, device_rects.ptr, device_depths.ptr,
             offsets.ptr, record_count, ids.ptr, tile_offsets.ptr, keys.ptr)
    context.synchronize()
    np.testing.assert_array_equal(tile_offsets.numpy(), expected_offsets)
    np.testing.assert_array_equal(ids.numpy()[:record_count], owner[order])
    expected_keys = tile[order].astype(np.uint64) << np.uint64(32) | depths[owner[order]].view(np.uint32)
    np.testing.assert_array_equal(keys.numpy()[:record_count], expected_keys)
