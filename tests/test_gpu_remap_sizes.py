"""The moments' copy on either side of the size (256 MB of old and new moments) from which it passes by the
caches, against a NumPy gather: equal bits, zeros for new Gaussians and parents out of range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 464 bytes a Gaussian: the line is at 578,524 old and new ones.
SIZES = [(1, 1), (0, 5), (100, 63), (63, 65), (289_262, 289_262), (289_262, 289_263), (200_000, 400_001)]


@pytest.mark.parametrize("previous,count", SIZES)
def test_remap(gsn, context, previous, count):
    rng = np.random.default_rng(count)
    parents = rng.integers(-1, max(previous, 1) + 2, count).astype(np.int32)
    first, second = (rng.normal(size=(58, max(previous, 1))).astype(np.float32) for _ in range(2))
    old, new = gsn.Moments.from_numpy(first, second), gsn.Moments(count)
    device_parents = gsn.DeviceBuffer.from_numpy(parents)
    gsn.call("gsn_remap_history", context.handle, device_parents.ptr, previous, count, old.ptr, new.ptr)
    context.synchronize()
    inherited = (parents >= 0) & (parents < previous)
    for got, source in zip(new.numpy(), (first, second)):
        expected = np.where(inherited, source[:, np.where(inherited, parents, 0)], np.float32(0.0))
        np.testing.assert_array_equal(got.view(np.uint32), expected.view(np.uint32))
