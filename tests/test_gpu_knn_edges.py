"""The 3-nearest-neighbour search around the sizes of its tree (leaves of 8 points, nodes of 8 boxes,
levels built in pairs) against the exhaustive oracle: indices and distances equal, also with
duplicates, where the smaller index wins, and with coordinates that are NaN (at no distance from
anything), infinite, or so large that distances are."""
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


@pytest.mark.parametrize("n", [2, 3, 4, 9, 65, 70, 700, 4097])
@pytest.mark.parametrize("kind", ["some nan", "nan in one axis", "infinite in one axis", "large", "all nan", "leaf of nan"])
def test_not_finite(gsn, context, oracle, n, kind):
    rng = np.random.default_rng(n + 1)
    points = rng.normal(size=(n, 3)).astype(np.float32)
    some = rng.random(n) < 0.2
    if kind == "some nan":
        points[some] = np.nan
    if kind == "nan in one axis":
        points[some, 1] = np.nan
    if kind == "infinite in one axis":
        points[some, 0] = np.where(rng.random(some.sum()) < 0.5, np.inf, -np.inf)
    if kind == "large":
        points *= np.float32(1e30)
    if kind == "all nan":
        points[:] = np.nan
    if kind == "leaf of nan":  # more than a leaf of them, at the end of the Morton order
        points[n // 2:] = np.nan
    neighbors, distances = gsn.knn3(context, points)
    expected_neighbors, expected = oracle.knn3(points)
    np.testing.assert_array_equal(neighbors, expected_neighbors)
    np.testing.assert_array_equal(distances.view(np.uint32), expected.view(np.uint32))
