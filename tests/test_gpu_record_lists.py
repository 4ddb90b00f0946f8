"""Tile lists of views whose list entries have few records for the screen's size (most Gaussians culled,
or splats of a tile or two), which sort their records, against a NumPy stable sort by (tile, depth, id):
record counts on either side of the line where the other way takes over (4 R = N times the 32x32-tile
parts of the screen), of the sort's 4,096-record tiles and of the 128 of them up to which its
scatter forms the digits' starts, long runs of entries without records, and record counts that are not
what the rectangles hold. Integers: equal."""
import numpy as np
import pytest

from test_gpu_tile_list_bounds import _check

pytestmark = pytest.mark.gpu

GRID = (120, 68)  # 12 parts


def _scene(count, records, grid=GRID, side=3, empty=0.0, seed=0):
    """`records` records in all: rectangles of up to side x side tiles, the rest culled or empty."""
    rng = np.random.default_rng(seed + count)
    width, height = rng.integers(1, side + 1, (2, count))
    x0 = (rng.random(count) ** 2 * (grid[0] - width + 1)).astype(np.int64)
    y0 = (rng.random(count) ** 2 * (grid[1] - height + 1)).astype(np.int64)
    visible = np.cumsum(width * height) <= records
    left = records - int((width * height)[visible].sum())
    for k in range(int(visible.sum()), int(visible.sum()) + left):  # single tiles up to the exact number
        width[k] = height[k] = 1
        visible[k] = True
    order = rng.permutation(count)
    rects = np.stack([x0, y0, x0 + width, y0 + height], axis=1)[order]
    visible = visible[order]
    rects[~visible] = -12345
    if empty:  # culled Gaussians that are in the list without a record
        some = ~visible & (rng.random(count) < empty)
        rects[some] = [3, 3, 3, 9]
        visible = visible | some
    return rects, rng.integers(1, 2 + count // 3, count).astype(np.float32), visible


@pytest.mark.parametrize("records", [1, 4095, 4096, 4097, 524_288, 524_289, 2_999_999, 3_000_000, 3_000_001])
def test_few_records(gsn, context, records):
    count = 1_000_000  # 12M tests: the line is at 3M records
    _check(gsn, context, GRID, *_scene(count, records), records)


@pytest.mark.parametrize("grid", [(64, 64), (65, 64), (1, 9000), (512, 511), (256, 256)])
def test_grids(gsn, context, grid):
    parts = -(-grid[0] // 32) * -(-grid[1] // 32)
    count = max(9_000_000 // parts, 40_000)
    side = 1 if grid[0] == 1 else 3
    _check(gsn, context, grid, *_scene(count, min(30_000, count // 4), grid, side), min(30_000, count // 4))


def test_entries_without_records(gsn, context):
    """More than 4,097 entries between two records: a block's owners do not fit its table."""
    _check(gsn, context, GRID, *_scene(1_000_000, 5000, empty=1.0), 5000)


@pytest.mark.parametrize("given", [1, 333, 50_000, 99_999, 100_001, 250_000])
def test_other_record_counts(gsn, context, given):
    _check(gsn, context, GRID, *_scene(1_000_000, 100_000, side=9), given)


def test_rectangles_of_a_larger_camera(gsn, context):
    rects, depths, visible = _scene(1_000_000, 60_000, (200, 200), 6)
    _check(gsn, context, GRID, rects, depths, visible, 60_000)


def test_more_records_than_31_bits(gsn, context):
    """1M rectangles of the whole 8,160-tile screen given as 700,001 records: 8.2e9 of them."""
    count = 1_000_000
    rects = np.tile(np.array([0, 0, *GRID]), (count, 1))
    depths = np.random.default_rng(1).permutation(count).astype(np.float32) + 1
    _check(gsn, context, GRID, rects, depths, np.ones(count, bool), 700_001)
