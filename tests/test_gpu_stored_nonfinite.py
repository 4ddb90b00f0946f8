"""The stored-state backward keeps what is not finite to the splats of its pixels: with a NaN or an
infinity in one pixel of the image gradient, or in one splat's colour, every Gaussian that no such
pixel blends has the gradients, bit for bit, that it has without. On either side of the tile count at
which a tile goes from four waves to one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BACKGROUND = (0.1, 0.2, 0.3)
COUNT = 250
REGION = 96  # the scene lies in the first rows and columns of the image


def _run(gsn, context, scenes, size):
    params = scenes.config0_params(seed=23, count=COUNT, sh_degree=0)
    params[0:2] *= np.float32(0.6)
    params[3:6] += np.float32(0.7)
    params[9] -= np.float32(1.0)  # nothing saturates: a pixel blends every splat that reaches it
    camera = gsn.Camera.make(size, size, 100.0, 100.0, 0.5 * REGION, 0.5 * REGION, None, [0.0, 0.0, 3.0])
    device = gsn.DeviceBuffer.from_numpy(params)
    image = gsn.DeviceBuffer((size, size, 3), np.float32)
    state = (gsn.DeviceBuffer((size, size), np.float32), gsn.DeviceBuffer((size, size), np.int32))
    projection = gsn.render(context, device, COUNT, camera, BACKGROUND, image, 0, stored_state=state)
    upstream = np.zeros((size, size, 3), np.float32)
    upstream[:REGION, :REGION] = np.random.default_rng(2).normal(size=(REGION, REGION, 3))
    return device, state, projection, upstream


def _gradients(gsn, context, run, upstream):
    device, state, projection, _ = run
    gradients, stats, absolute = (gsn.DeviceBuffer((k, COUNT), np.float32) for k in (58, 2, 2))
    device_upstream = gsn.DeviceBuffer.from_numpy(upstream)
    gsn.gaussian_gradients_stored(context, projection, device, 0, *state, BACKGROUND, device_upstream, gradients, stats,
                                  absolute)
    context.synchronize()
    return gradients.numpy()


def _reached(projection):
    """[Gaussian, row, column] of the region: alpha at or above 1% below its threshold."""
    means = projection.means.numpy()[:COUNT].astype(np.float64)
    a, b, c, opacity = projection.conic_opacities.numpy()[:COUNT].astype(np.float64).T[:, :, None, None]
    visible = np.diff(projection.record_offsets.numpy()) > 0
    rows, columns = np.mgrid[:REGION, :REGION]
    dx, dy = means[:, 0, None, None] - columns, means[:, 1, None, None] - rows
    alpha = opacity * np.exp(-0.5 * (a * dx * dx + c * dy * dy) - b * dx * dy)
    return (alpha >= 0.99 / 255.0) & visible[:, None, None]


def _check(clean, spoiled, affected):
    assert np.isfinite(clean).all()
    np.testing.assert_array_equal(spoiled[:, ~affected].view(np.uint32), clean[:, ~affected].view(np.uint32))


@pytest.mark.parametrize("size", [REGION, 16 * 56])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_gradient_of_one_pixel(gsn, context, scenes, size, value):
    run = _run(gsn, context, scenes, size)
    reached = _reached(run[2])
    clean = _gradients(gsn, context, run, run[3])
    tested = 0
    for row, column in ((40, 44), (53, 50), (61, 33)):
        upstream = run[3].copy()
        upstream[row, column, 1] = value
        spoiled = _gradients(gsn, context, run, upstream)
        affected = reached[:, row, column]
        _check(clean, spoiled, affected)
        assert not np.isfinite(spoiled[:, affected]).all()
        # Gaussians that blend beside the pixel, in its band of the tile, and not at it.
        band = reached[:, row // 4 * 4:row // 4 * 4 + 4, column // 16 * 16:column // 16 * 16 + 16].any(axis=(1, 2))
        tested += (band & ~affected).sum()
    assert tested > 10


@pytest.mark.parametrize("size", [REGION, 16 * 56])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_colour_of_one_splat(gsn, context, scenes, size, value):
    run = _run(gsn, context, scenes, size)
    projection = run[2]
    reached = _reached(projection)
    clean = _gradients(gsn, context, run, run[3])
    colours = projection.colors.numpy()
    tested = 0
    areas = reached.sum(axis=(1, 2))
    for splat in np.argsort(np.where(areas > 20, areas, 1 << 30))[:6]:
        spoiled_colours = colours.copy()
        spoiled_colours[splat, 0] = value
        projection.colors.upload(spoiled_colours)
        spoiled = _gradients(gsn, context, run, run[3])
        affected = (reached & reached[splat]).any(axis=(1, 2))
        _check(clean, spoiled, affected)
        tested += (~affected & (reached & _bands_of(reached[splat])).any(axis=(1, 2))).sum()
    projection.colors.upload(colours)
    assert tested > 10


def _bands_of(pixels):
    """The 16x4-pixel bands that hold any of the pixels."""
    bands = pixels.reshape(REGION // 4, 4, REGION // 16, 16).any(axis=(1, 3))
    return bands.repeat(4, axis=0).repeat(16, axis=1)
