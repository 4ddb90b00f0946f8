"""The rasterisers split a tile over one, two or four waves by the number of tiles of the image.
One scene is drawn into canvases of growing size with the same focal length and principal point:
the shared corner of the images must be equal bit for bit, whatever the split, and gradients of a
loss on that corner may differ only by the order of the sums over a record's pixels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CORNER = (61, 83)  # rows, columns: not multiples of the 16-pixel tile nor of the 4-row band
# Tiles on either side of each boundary of the rules (3,072 and 9,600), more, and one row of tiles.
CANVASES = [(61, 83), (768, 1024), (768, 1040), (1536, 1600), (1536, 1616), (1536, 2048), (1536, 2064), (16 * 3073, 16)]


def _draw(gsn, context, scenes, canvas, stored):
    height, width = canvas
    params = scenes.config0_params(seed=31, count=700, sh_degree=2)
    params[0:2] *= np.float32(0.25)  # inside every canvas's view, away from the field-of-view clamp
    params[3:6] += np.float32(0.8)
    params[9] += np.float32(1.0)  # some pixels saturate
    camera = gsn.Camera.make(width, height, 90.0, 90.0, 7.5 if width == 16 else 40.0, 30.0, None, [0.0, 0.0, 3.0])
    device = gsn.DeviceBuffer.from_numpy(params)
    image = gsn.DeviceBuffer((height, width, 3), np.float32)
    state = (gsn.DeviceBuffer((height, width), np.float32), gsn.DeviceBuffer((height, width), np.int32))
    projection = gsn.render(context, device, params.shape[1], camera, (0.2, 0.4, 0.1), image, 2,
                            stored_state=state if stored else None)
    rows, columns = CORNER[0], min(CORNER[1], width)
    upstream = np.zeros((height, width, 3), np.float32)
    upstream[:rows, :columns] = np.random.default_rng(5).normal(size=(CORNER[0], CORNER[1], 3))[:, :columns]
    gradients, stats, absolute = (gsn.DeviceBuffer((k, params.shape[1]), np.float32) for k in (58, 2, 2))
    if stored:
        gsn.gaussian_gradients_stored(context, projection, device, 2, *state, (0.2, 0.4, 0.1),
                                      gsn.DeviceBuffer.from_numpy(upstream), gradients, stats, absolute)
    else:
        gsn.gaussian_gradients(context, projection, device, 2, image, gsn.DeviceBuffer.from_numpy(upstream),
                               gradients, stats, absolute)
    context.synchronize()
    return image.numpy()[:rows, :columns], gradients.numpy()


@pytest.mark.parametrize("stored", [False, True])
@pytest.mark.parametrize("canvas", CANVASES[1:])
def test_split_does_not_change_the_result(gsn, context, scenes, canvas, stored):
    small = CANVASES[0] if canvas[1] > 16 else (61, 16)
    image, gradients = _draw(gsn, context, scenes, small, stored)
    other_image, other_gradients = _draw(gsn, context, scenes, canvas, stored)
    np.testing.assert_array_equal(other_image, image)
    assert np.abs(gradients).max() > 0
    for row in range(58):
        scale = np.linalg.norm(gradients[row].astype(np.float64))
        error = np.linalg.norm(other_gradients[row].astype(np.float64) - gradients[row])
        assert error <= 1e-5 * scale, f"row {row}: {error / max(scale, 1e-30):.2e}"
