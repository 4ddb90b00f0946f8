"""The 3-nearest-neighbour search around the sizes of its tree (leaves of 8 points, nodes of 8 boxes,
levels built in pairs) against the exhaustive oracle: indices and distances equal, also with
duplicates, where the smaller index wins."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 4, 5, 7, 8, 9, 63, 64, 65, 511, 512, 513, 4095, 4096, 4097, 9000])
@pytest.mark.parametrize("kind", ["uniform", "clusters", "duplicates"])
def test_knn(gsn, context, oracle, n, kind):
    rng = np.random.default_rng(n)
    points = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    if kind == "clusters":  # few far points among many close ones
        points[n // 20:] *= np.float32(1e-3)
    if kind == "duplicates":
        points = np.round(points * np.float32(4.0))
    neighbors, distances = gsn.knn3(context, points)
    expected_neighbors, expected = oracle.knn3(points)
    np.testing.assert_array_equal(neighbors, expected_neighbors)
    np.testing.assert_array_equal(distances.view(np.uint32), expected.view(np.uint32))
