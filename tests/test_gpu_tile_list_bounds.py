"""gsn_build_tile_lists when its record count is not what the rectangles hold: a buffer of fixed
capacity, a stale count, rectangles of another camera. The lists then hold the first record_count
records of the rectangles inside the grid, nearest first and row by row inside a rectangle; every
offset stays within the record count, every id below the last offset is written and nothing past the
record count is. Integers: equal."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GUARD = 64
UNWRITTEN = -77


def _build(gsn, context, grid, rects, depths, visible, record_count):
    """(offsets, ids, keys) with GUARD entries past their ends that must keep their value."""
    tiles = grid[0] * grid[1]
    camera = gsn.Camera.make(16 * grid[0], 16 * grid[1], 1.0, 1.0, 0.0, 0.0)
    device = [gsn.DeviceBuffer.from_numpy(a) for a in (
        rects.astype(np.int32), depths, np.concatenate([[0], np.cumsum(visible)]).astype(np.int32))]
    ids = gsn.DeviceBuffer.from_numpy(np.full(record_count + GUARD, UNWRITTEN, np.int32))
    keys = gsn.DeviceBuffer.from_numpy(np.full(record_count + GUARD, 5, np.uint64))
    offsets = gsn.DeviceBuffer.from_numpy(np.full(tiles + 1 + GUARD, UNWRITTEN, np.int64))
    gsn.call("gsn_build_tile_lists", context.handle, ctypes.byref(camera), len(depths), device[0].ptr, device[1].ptr,
             device[2].ptr, record_count, ids.ptr, offsets.ptr, keys.ptr)
    context.synchronize()
    ids, keys, offsets = ids.numpy(), keys.numpy(), offsets.numpy()
    assert (ids[record_count:] == UNWRITTEN).all() and (keys[record_count:] == 5).all()
    assert (offsets[tiles + 1:] == UNWRITTEN).all()
    return offsets[:tiles + 1], ids[:record_count], keys[:record_count]


def _check(gsn, context, grid, rects, depths, visible, record_count):
    order = np.argsort(depths, kind="stable")
    order = order[visible[order]]
    r = np.clip(rects[order], 0, [grid[0], grid[1], grid[0], grid[1]])
    width, height = np.maximum(r[:, 2] - r[:, 0], 0), np.maximum(r[:, 3] - r[:, 1], 0)
    ends = np.cumsum(width * height)
    used = min(int(np.searchsorted(ends, record_count)) + 1, len(order))  # entries that reach the lists
    order, r, width, areas = order[:used], r[:used], width[:used], (width * height)[:used]
    owner = np.repeat(np.arange(used), areas)
    local = np.arange(len(owner)) - (np.cumsum(areas) - areas)[owner]
    tile = ((r[owner, 1] + local // np.maximum(width[owner], 1)) * grid[0] + r[owner, 0] + local % np.maximum(width[owner], 1))
    tile, owner = tile[:record_count], order[owner[:record_count]]
    by_tile = np.argsort(tile, kind="stable")
    tile, owner = tile[by_tile], owner[by_tile]

    offsets, ids, keys = _build(gsn, context, grid, rects, depths, visible, record_count)
    assert offsets[0] == 0 and offsets[-1] == len(tile) and (np.diff(offsets) >= 0).all()
    np.testing.assert_array_equal(offsets, np.searchsorted(tile, np.arange(grid[0] * grid[1] + 1)))
    np.testing.assert_array_equal(ids[:len(tile)], owner)
    np.testing.assert_array_equal(keys[:len(tile)],
                                  tile.astype(np.uint64) << np.uint64(32) | depths[owner].view(np.uint32))
    assert (keys[len(tile):] == np.uint64(0xffffffffffffffff)).all()


def _scene(grid, count, side, seed, culled=0.1):
    rng = np.random.default_rng(seed)
    width, height = rng.integers(1, min(side, grid[0]) + 1, count), rng.integers(1, min(side, grid[1]) + 1, count)
    x0 = (rng.random(count) ** 2 * (grid[0] - width + 1)).astype(np.int64)
    y0 = (rng.random(count) ** 2 * (grid[1] - height + 1)).astype(np.int64)
    rects = np.stack([x0, y0, x0 + width, y0 + height], axis=1)
    visible = rng.random(count) >= culled
    visible[0] = True
    rects[~visible] = -12345
    return rects, rng.integers(1, 2 + count // 3, count).astype(np.float32), visible


# Small and large grids, chunks of 256 entries and of thousands, entries without records.
SCENES = [((1, 1), 40, 1, 0.1), ((7, 5), 300, 5, 0.1), ((33, 32), 4097, 12, 0.1), ((64, 40), 5000, 40, 0.1),
          ((120, 68), 60_000, 9, 0.6), ((40, 33), 400_000, 3, 0.1)]


@pytest.mark.parametrize("grid,count,side,culled", SCENES)
@pytest.mark.parametrize("kept", ["one", "third", "all but one", "all", "one more", "twice"])
def test_other_record_counts(gsn, context, grid, count, side, culled, kept):
    rects, depths, visible = _scene(grid, count, side, count, culled)
    held = int(((rects[:, 2] - rects[:, 0]) * (rects[:, 3] - rects[:, 1]))[visible].sum())
    record_count = {"one": 1, "third": held // 3 + 1, "all but one": max(held - 1, 1), "all": held,
                    "one more": held + 1, "twice": 2 * held}[kept]
    _check(gsn, context, grid, rects, depths, visible, record_count)


@pytest.mark.parametrize("rects_grid,grid", [((64, 40), (20, 33)), ((20, 33), (64, 40)), ((64, 40), (64, 9))])
@pytest.mark.parametrize("share", [0.4, 1.0])
def test_rectangles_of_another_camera(gsn, context, rects_grid, grid, share):
    rects, depths, visible = _scene(rects_grid, 5000, 12, 3)
    held = int(((rects[:, 2] - rects[:, 0]) * (rects[:, 3] - rects[:, 1]))[visible].sum())
    _check(gsn, context, grid, rects, depths, visible, int(share * held))


def test_more_records_than_32_bits(gsn, context):
    """20,000 rectangles of the whole 512x511-tile screen: 5.2e9 records."""
    grid, count = (512, 511), 20_000
    rects = np.tile(np.array([0, 0, *grid]), (count, 1))
    depths = np.random.default_rng(1).permutation(count).astype(np.float32) + 1
    _check(gsn, context, grid, rects, depths, np.ones(count, bool), 1_300_001)


def test_cut_lists_render(gsn, context, scenes):
    """A render from lists cut at a third draws the picture of the Gaussians that they hold."""
    params = scenes.config0_params(seed=5, count=3000, sh_degree=0)
    camera = gsn.Camera.make(160, 112, 120.0, 120.0, 79.5, 55.5, None, [0.0, 0.0, 3.0])
    images = [gsn.DeviceBuffer((112, 160, 3), np.float32) for _ in range(2)]
    device_params = gsn.DeviceBuffer.from_numpy(params)
    p = gsn.render(context, device_params, 3000, camera, (0.1, 0.2, 0.3), images[0], 0)
    full = images[0].numpy()
    third = p.record_count // 3
    call = lambda n: gsn.call("gsn_build_tile_lists", context.handle, ctypes.byref(camera), 3000, p.tile_rects.ptr,
                              p.depths.ptr, p.record_offsets.ptr, n, p.tile_gaussian_ids.ptr, p.tile_offsets.ptr, None)
    call(third)
    background = (ctypes.c_float * 3)(0.1, 0.2, 0.3)
    gsn.call("gsn_render_tiles", context.handle, ctypes.byref(camera), p.tile_gaussian_ids.ptr, p.tile_offsets.ptr,
             p.means.ptr, p.conic_opacities.ptr, p.colors.ptr, background, images[1].ptr)
    context.synchronize()
    cut = images[1].numpy()
    assert np.isfinite(cut).all() and not np.array_equal(cut, full)
    offsets = p.tile_offsets.numpy()
    assert offsets[-1] == third
    # Only tiles whose lists were cut differ.
    call(p.record_count)
    context.synchronize()
    shorter = np.diff(offsets) < np.diff(p.tile_offsets.numpy())
    changed = (cut != full).any(axis=2).reshape(7, 16, 10, 16).any(axis=(1, 3)).ravel()
    assert not (changed & ~shorter).any()
