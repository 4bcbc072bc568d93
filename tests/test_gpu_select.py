"""Selection over key rows (the k smallest by key and column) through the public searches: rows
shorter than a workgroup, ties beyond the selection's buffer, long rows cut into segments, and
the route of small default searches against the fused tile."""
import numpy as np
import pytest

import aoclda

pytestmark = pytest.mark.gpu


def check(oracle, X, Q, k, metric="euclidean", **kw):
    nn = aoclda.neighbors.nearest_neighbors(metric=metric, **kw).fit(X)
    dist, ind = nn.kneighbors(Q, n_neighbors=k)
    ei, ed = oracle.knn(X.astype(np.float64), Q.astype(np.float64), k, metric)
    np.testing.assert_array_equal(ind, ei)
    # Exact distances, rounded once to the type.
    np.testing.assert_allclose(dist, ed, rtol=1e-12 if X.dtype == np.float64 else 1e-6,
                               atol=1e-12)
    return ind


# 255-257: one element per thread or fewer; 2,047-2,049: the unrolled sweep's edges.
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 31, 255, 256, 257, 2047, 2049, 5000])
@pytest.mark.parametrize("k", [1, 5, 100, 128, 129])
def test_small_searches(oracle, dtype, n, k):
    if k > n:
        pytest.skip("k > n")
    rng = np.random.default_rng(n * 131 + k)
    X = rng.standard_normal((n, 7)).astype(dtype)
    Q = rng.standard_normal((33, 7)).astype(dtype)
    ind = check(oracle, X, Q, k)
    if k <= 128 and n >= 16:
        # The same search on the fused tile.
        np.testing.assert_array_equal(check(oracle, X, Q, k, tile_variant=3), ind)


@pytest.mark.parametrize("k", [3, 128])
def test_ties_beyond_the_buffer(oracle, k):
    """Thousands of equal keys at the bound: the general selection takes those rows over and
    keeps the lowest columns."""
    X = np.zeros((6000, 3))
    X[::7] = 1.0
    Q = np.vstack([np.zeros((3, 3)), np.ones((2, 3)), np.full((2, 3), 0.5)])
    check(oracle, X, Q, k)


@pytest.mark.parametrize("metric", ["manhattan", "cosine", "inner_product"])
@pytest.mark.parametrize("n", [40000, 70001])
def test_long_rows_in_segments(oracle, metric, n):
    """Few queries against many rows: the keys of a row are selected from in segments, ties
    (duplicated rows in different segments) by column."""
    rng = np.random.default_rng(n)
    X = rng.integers(-3, 4, (n, 5)).astype(np.float64)
    X[:, 0] += 0.5
    Q = rng.integers(-3, 4, (3, 5)).astype(np.float64) + 0.25
    nn = aoclda.neighbors.nearest_neighbors(metric=metric).fit(X)
    dist, ind = nn.kneighbors(Q, n_neighbors=50)
    if metric == "manhattan":
        key = np.abs(X[None] - Q[:, None]).sum(-1)
    elif metric == "inner_product":
        key = -(Q @ X.T)
    else:
        key = 1.0 - (Q @ X.T) / (np.linalg.norm(Q, axis=1)[:, None] * np.linalg.norm(X, axis=1))
    if metric == "cosine":
        # Rounding may order equal cosines either way: the distances decide.
        np.testing.assert_allclose(dist, np.sort(key, axis=1)[:, :50], rtol=0, atol=1e-14)
    else:  # sums of multiples of 1/4: exact
        np.testing.assert_array_equal(ind, np.argsort(key, axis=1, kind="stable")[:, :50])
