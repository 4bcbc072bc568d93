"""kNN of rows wider than the fused tile and of the cosine metric (approximate scores on the
matrix cores, exact keys, certification) against the oracle: tile edges, odd widths, both types,
and the data that end in the exact fallback or the general path."""
import ctypes as C

import numpy as np
import pytest

import aoclda
from aoclda import _lib as L

pytestmark = pytest.mark.gpu


def stats(nn):
    nfb, ncand = L.da_int(), L.da_int()
    L.check(L.lib.da_nn_last_query_stats(nn.handle.h, C.byref(nfb), C.byref(ncand)))
    return nfb.value, ncand.value


def search(oracle, X, Q, k, metric, wide=True):
    nn = aoclda.neighbors.nearest_neighbors(metric=metric, algorithm="brute").fit(X)
    dist, ind = nn.kneighbors(Q, n_neighbors=k)
    nfb, ncand = stats(nn)
    assert (ncand > 0) == wide
    ei, ed = oracle.knn(X.astype(np.float64), Q.astype(np.float64), k, metric)
    if metric == "cosine":
        # 1 - x.y / (|x||y|) carries a few 2^-53 either side: equal cosines may swap.
        np.testing.assert_allclose(dist, ed, rtol=0, atol=1e-6 if X.dtype == np.float32 else 1e-14)
        assert (ind == ei).mean() > 0.999
    else:
        np.testing.assert_array_equal(ind, ei)
        np.testing.assert_allclose(dist, ed, rtol=1e-6 if X.dtype == np.float32 else 1e-12,
                                   atol=1e-12)
    return nfb


def mixture(rng, n, d, dtype, offset=0.0):
    means = rng.uniform(-10, 10, (8, d)) + offset
    return (means[rng.integers(0, 8, n)] + rng.standard_normal((n, d))).astype(dtype)


# 128-row tiles, k steps of 32 features (odd and even counts), blocks of 256 features.
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,nq,d,k", [(4096, 4100, 129, 5), (5001, 3300, 160, 32),
                                      (8321, 1025, 255, 33), (4097, 2049, 257, 96),
                                      (6000, 900, 511, 1), (3000, 1000, 784, 10)])
@pytest.mark.parametrize("metric", ["euclidean", "sqeuclidean", "cosine"])
def test_wide(oracle, dtype, n, nq, d, k, metric):
    rng = np.random.default_rng(n + d)
    X = mixture(rng, n, d, dtype)
    Q = mixture(rng, nq, d, dtype)
    Q[:5] = X[:5]
    search(oracle, X, Q, k, metric)


@pytest.mark.parametrize("d", [2, 16, 100])
def test_cosine_narrow(oracle, d):
    rng = np.random.default_rng(d)
    n = (1 << 31) // (d * 3000) + 1
    if n * 3000 * 8 > 2 ** 34:
        n, nq = 400000, 1 + (1 << 31) // (d * 400000)
    else:
        nq = 3000
    X = mixture(rng, n, d, np.float32)
    Q = mixture(rng, nq, d, np.float32)
    Q, X[7] = Q[:nq], 0.0  # a zero row: norm taken as 1
    nn = aoclda.neighbors.nearest_neighbors(metric="cosine", algorithm="brute").fit(X)
    dist, ind = nn.kneighbors(Q, n_neighbors=4)
    X64, Q64 = X.astype(np.float64), Q[:40].astype(np.float64)
    nx, nq_ = np.linalg.norm(X64, axis=1), np.linalg.norm(Q64, axis=1)
    nx[7] = 1.0
    key = 1.0 - (Q64 @ X64.T) / (nq_[:, None] * nx)
    np.testing.assert_allclose(dist[:40], np.sort(key, axis=1)[:, :4], rtol=1e-5, atol=1e-12)


@pytest.mark.parametrize("case", ["offset", "duplicates", "query_out_of_range", "outlier",
                                  "nonfinite", "query_nan"])
def test_data(oracle, case):
    """Far from the origin, ties beyond the candidate list (exact fallback), queries beyond the
    operand range (exact fallback), an outlier that swamps the scale, and training values that are
    not finite (the general path)."""
    rng = np.random.default_rng(3)
    n, nq, d = 4500, 2600, 192
    X, Q = mixture(rng, n, d, np.float32), mixture(rng, nq, d, np.float32)
    wide, expect_fallback = True, False
    if case == "offset":
        X, Q = X + np.float32(5000), Q + np.float32(5000)
    elif case == "duplicates":
        X = X[rng.integers(0, 20, n)]
        expect_fallback = True
    elif case == "query_out_of_range":
        Q[11] = 1e6
        expect_fallback = True
    elif case == "outlier":
        X[5] = 1e7
        expect_fallback = True
    elif case == "nonfinite":
        X[5, 3] = np.inf
        wide = False
    elif case == "query_nan":
        Q[4, 0] = np.nan
        expect_fallback = True
    if case == "nonfinite":
        # The row at infinity is never a neighbour; the rest are as without it.
        nn = aoclda.neighbors.nearest_neighbors(algorithm="brute").fit(X)
        dist, ind = nn.kneighbors(Q, n_neighbors=5)
        assert stats(nn)[1] == 0
        keep = np.delete(np.arange(n), 5)
        ei, ed = oracle.knn(X[keep].astype(np.float64), Q.astype(np.float64), 5)
        np.testing.assert_array_equal(ind, keep[ei])
        return
    if case == "query_nan":
        nn = aoclda.neighbors.nearest_neighbors(algorithm="brute").fit(X)
        dist, ind = nn.kneighbors(Q, n_neighbors=5)
        ok = np.delete(np.arange(nq), 4)
        ei, ed = oracle.knn(X.astype(np.float64), Q[ok].astype(np.float64), 5)
        np.testing.assert_array_equal(ind[ok], ei)
        assert stats(nn)[0] >= 1
        return
    nfb = search(oracle, X, Q, 5, "euclidean", wide)
    if expect_fallback:
        assert nfb > 0


@pytest.mark.parametrize("where", ["rows", "queries"])
@pytest.mark.parametrize("d", [16, 160])
def test_cosine_norms_that_overflow(oracle, d, where):
    """Rows of 1e200 have infinite norms: products with ordinary rows give the key 1, with large
    ones infinity over infinity, which comes last. Key tiles in slices that are too small for the
    approximate scores are the answer."""
    rng = np.random.default_rng(d)
    n, nq, k = 40000 if d == 16 else 5000, 3600 if d == 16 else 2800, 90
    X, Q = rng.standard_normal((n, d)), rng.standard_normal((nq, d))
    X[:, 0] -= 50  # most rows point away from the queries
    Q[:, 0] += 50
    X[::n // 9, 0] += 100
    if where == "rows":
        X[5::n // 30] *= 1e200
        Q *= 1e150
    else:
        Q[::7] *= 1e200
    nn = aoclda.neighbors.nearest_neighbors(metric="cosine", algorithm="brute").fit(X)
    dist, ind = nn.kneighbors(Q, n_neighbors=k)
    for i in range(0, nq, 400):
        de, ie = nn.kneighbors(Q[i:i + 400], n_neighbors=k)
        assert stats(nn)[1] == 0  # the general path
        np.testing.assert_array_equal(ind[i:i + 400], ie)
        np.testing.assert_array_equal(dist[i:i + 400], de)


@pytest.mark.parametrize("metric,d,nq", [("cosine", 16, 389), ("euclidean", 160, 389)])
def test_several_blocks(metric, d, nq):
    """Blocks of 128 queries and a ragged last one, some queries of each block beyond fp16's range;
    slices too small for the approximate scores are the answer."""
    rng = np.random.default_rng(d)
    n = 400000 if d == 16 else 300000
    X, Q = mixture(rng, n, d, np.float32), mixture(rng, nq, d, np.float32)
    Q[[3, 130, 300, 388]] *= 3000
    step = 250 if d == 16 else 40
    nn = aoclda.neighbors.nearest_neighbors(metric=metric, algorithm="brute").fit(X)
    dist, ind = nn.kneighbors(Q, n_neighbors=6)
    nfb, ncand = stats(nn)
    assert ncand > 0 and nfb < nq // 10
    for i in range(0, nq, step):
        de, ie = nn.kneighbors(Q[i:i + step], n_neighbors=6)
        assert stats(nn)[1] == 0
        np.testing.assert_array_equal(ind[i:i + step], ie)
        np.testing.assert_array_equal(dist[i:i + step], de)


def test_tight_clusters_are_not_tried_every_time():
    """Where most queries are searched again, the next searches take the key tiles at once."""
    rng = np.random.default_rng(4)
    means = rng.uniform(-10, 10, (8, 200))
    X = (means[rng.integers(0, 8, 9000)] + 1e-3 * rng.standard_normal((9000, 200))).astype(np.float32)
    Q = (means[rng.integers(0, 8, 1300)] + 1e-3 * rng.standard_normal((1300, 200))).astype(np.float32)
    nn = aoclda.neighbors.nearest_neighbors(algorithm="brute").fit(X)
    got = []
    for _ in range(4):
        got.append(nn.kneighbors(Q, n_neighbors=5) + stats(nn))
    assert [g[3] > 0 for g in got] == [True, False, True, False]
    assert got[0][2] > len(Q) // 2
    for g in got[1:]:
        np.testing.assert_array_equal(g[1], got[0][1])
        np.testing.assert_array_equal(g[0], got[0][0])
