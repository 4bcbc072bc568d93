"""kNN by hit bits (large searches of up to 128 features, squared-euclidean metrics): bit for bit the
neighbours of the fused tile (which serves a handle with a tile option set), and of the oracle. The
fused tile also serves the queries that the bits list, so tests on ordinary data bound their number."""
import ctypes as C

import numpy as np
import pytest

import aoclda
from aoclda import _lib as L

pytestmark = pytest.mark.gpu

KEEP = 2048  # hits per query; reported as the candidates of such a search


def _stats(nn):
    nfb, ncand = L.da_int(), L.da_int()
    L.check(L.lib.da_nn_last_query_stats(nn.handle.h, C.byref(nfb), C.byref(ncand)))
    return nfb.value, ncand.value


def _compare(X, Q, k, most_listed=None, **opts):
    nn = aoclda.neighbors.nearest_neighbors(**opts).fit(X)
    dist, ind = nn.kneighbors(Q, n_neighbors=k)
    nfb, ncand = _stats(nn)
    assert ncand == KEEP
    if most_listed is not None:
        assert nfb <= most_listed
    tile = aoclda.neighbors.nearest_neighbors(seed_thresholds=False, **opts).fit(X)
    de, ie = tile.kneighbors(Q, n_neighbors=k)
    assert _stats(tile)[1] != KEEP
    np.testing.assert_array_equal(ind, ie)
    np.testing.assert_array_equal(dist, de)
    return nfb


def _mixture(rng, n, d, dtype, means):
    return (means[rng.integers(0, len(means), n)] + rng.standard_normal((n, d))).astype(dtype)


def _queries(n, d):
    """Enough for the products from which searches take the hit bits, and ragged."""
    return int(np.ceil(2**32 / (n * (d + 16)))) + 37


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", [3, 31, 32, 33, 64, 65, 96, 97, 127, 128])
def test_widths(dtype, d):
    """One to four k steps and their edges; rows of whole 16-byte pieces and others."""
    rng = np.random.default_rng(d)
    means = rng.uniform(-10, 10, (16, d))
    X = _mixture(rng, 20011, d, dtype, means)
    Q = _mixture(rng, _queries(20011, d), d, dtype, means)
    # fewer than one query in ten is left to the tile, except in the few dimensions where a
    # cluster is dense against fp16's steps
    _compare(X, Q, 10, most_listed=len(Q) // 10 if d >= 31 else None)


@pytest.mark.parametrize("k", [1, 2, 20, 100, 128])
@pytest.mark.parametrize("n", [16384, 16385, 65537, 140000])
def test_sizes(n, k):
    rng = np.random.default_rng(n + k)
    means = rng.uniform(-10, 10, (8, 24))
    X = _mixture(rng, n, 24, np.float32, means)
    Q = _mixture(rng, _queries(n, 24), 24, np.float32, means)
    _compare(X, Q, k)


@pytest.mark.parametrize("precision", ["fp16", "fp16c", "bf16", "fp16x3"])
@pytest.mark.parametrize("metric", ["euclidean", "sqeuclidean", "euclidean_gemm", "sqeuclidean_gemm"])
def test_forms(precision, metric):
    rng = np.random.default_rng(3)
    means = rng.uniform(-10, 10, (8, 40))
    X = _mixture(rng, 30000, 40, np.float32, means)
    Q = _mixture(rng, 2600, 40, np.float32, means)
    _compare(X, Q, 12, precision=precision, metric=metric)


def test_difficult_queries():
    """Duplicates (ties by index), queries equal to rows, far queries, a value outside fp16's range,
    more equal rows than the merge holds."""
    rng = np.random.default_rng(7)
    means = rng.uniform(-10, 10, (8, 32))
    X = _mixture(rng, 40000, 32, np.float32, means)
    X[20000:20400] = X[:400]
    X[30000:33000] = X[5]
    Q = _mixture(rng, _queries(40000, 32), 32, np.float32, means)
    Q[:500] = X[:500]
    Q[600:620] *= 50
    Q[700] = 1e6  # beyond fp16 at the data's scale, its keys still distinct in double
    Q[701] = 0
    assert _compare(X, Q, 9) > 0


@pytest.mark.parametrize("scale,shift", [(1e-12, 0), (1e12, 0), (1e-3, 1e4)])
def test_ranges_and_tight_clusters(scale, shift):
    """Any magnitude; clusters so tight against their spread that fp16 cannot tell their rows apart
    (the sample shows it and the tile serves the search)."""
    rng = np.random.default_rng(11)
    means = rng.uniform(-10, 10, (8, 20))
    X = _mixture(rng, 30000, 20, np.float64, means) * scale + shift
    Q = _mixture(rng, 4100, 20, np.float64, means) * scale + shift
    _compare(X, Q, 5)
    X = means[rng.integers(0, 8, 30000)] + 1e-4 * rng.standard_normal((30000, 20))
    Q = means[rng.integers(0, 8, 4100)] + 1e-4 * rng.standard_normal((4100, 20))
    assert _compare(X, Q, 5) == len(Q)


def test_not_finite_rows():
    """A row so large that fp16 cannot hold the others beside it: the bits list every query."""
    rng = np.random.default_rng(13)
    X = rng.standard_normal((20000, 20)).astype(np.float32)
    X[77, 3] = 1e38
    Q = rng.standard_normal((6100, 20)).astype(np.float32)
    nn = aoclda.neighbors.nearest_neighbors().fit(X)
    dist, ind = nn.kneighbors(Q, n_neighbors=5)
    tile = aoclda.neighbors.nearest_neighbors(seed_thresholds=False).fit(X)
    de, ie = tile.kneighbors(Q, n_neighbors=5)
    np.testing.assert_array_equal(ind, ie)
    np.testing.assert_array_equal(dist, de)


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert L.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_blocks_and_workspaces(oracle):
    """Several query blocks and a ragged last one, with queries left to the tile in each: the
    results are those of the queries in slices of one block, and of the oracle. Few rows and many
    queries: the columns of the hits, 8 KB a query, are what fills a block's 1 GiB."""
    rng = np.random.default_rng(17)
    means = rng.uniform(-10, 10, (16, 16))
    X = _mixture(rng, 8192, 16, np.float32, means)
    Q = _mixture(rng, 300007, 16, np.float32, means)
    odd = [5, 120000, 239999, 300006]
    Q[odd] *= 500  # beyond fp16's range at the data's scale
    nn = aoclda.neighbors.nearest_neighbors().fit(X)
    nn.kneighbors(Q[:8192], n_neighbors=7)
    free = _free_bytes()
    dist, ind = nn.kneighbors(Q, n_neighbors=7)
    # workspaces, and the queries (19 MB) and results (17 MB) of a search on host arrays
    assert free - _free_bytes() < (1 << 30) + (64 << 20)
    nfb, ncand = _stats(nn)
    assert ncand == KEEP and len(odd) <= nfb < 30000
    for i in range(0, len(Q), 90000):
        de, ie = nn.kneighbors(Q[i:i + 90000], n_neighbors=7)
        np.testing.assert_array_equal(ind[i:i + 90000], ie)
        np.testing.assert_array_equal(dist[i:i + 90000], de)
    pick = np.concatenate([odd, rng.integers(0, len(Q), 500)])
    ei, ed = oracle.knn(X.astype(np.float64), Q[pick].astype(np.float64), 7)
    np.testing.assert_array_equal(ind[pick], ei)
    np.testing.assert_allclose(dist[pick], ed, rtol=1.2e-7)  # one rounding to float


@pytest.mark.parametrize("n", [8192, 20000, 30000])
def test_tight_clusters_are_not_tried_every_time(n):
    """Clusters that fp16 cannot resolve hold thousands of hits a query: the sample shows it at
    any number of rows (every query is listed before the sweep), and of the searches that follow
    1, 2, 4, ... go straight to the fused tile before the bits are tried again."""
    rng = np.random.default_rng(n)
    means = rng.uniform(-10, 10, (2, 20))
    X = means[rng.integers(0, 2, n)] + 1e-4 * rng.standard_normal((n, 20))
    Q = means[rng.integers(0, 2, 6000)] + 1e-4 * rng.standard_normal((6000, 20))
    nn = aoclda.neighbors.nearest_neighbors().fit(X)
    tile = aoclda.neighbors.nearest_neighbors(seed_thresholds=False).fit(X)
    de, ie = tile.kneighbors(Q, n_neighbors=5)
    tried = []
    for _ in range(6):
        dist, ind = nn.kneighbors(Q, n_neighbors=5)
        np.testing.assert_array_equal(ind, ie)
        np.testing.assert_array_equal(dist, de)
        nfb, ncand = _stats(nn)
        tried.append(ncand == KEEP)
        assert not tried[-1] or nfb == len(Q)
    assert tried == [True, False, True, False, False, True]
    # new training rows are tried at once, and stay with the bits
    X = rng.uniform(-10, 10, (n, 20))
    nn.fit(X)
    for _ in range(3):
        nn.kneighbors(X[:6000], n_neighbors=5)
        assert _stats(nn)[1] == KEEP and _stats(nn)[0] < 600


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_nan_and_infinity(dtype):
    """Training rows that are not finite keep the search on the tile's path; queries that are not
    finite are listed and come out as the tile's, the others untouched by them."""
    rng = np.random.default_rng(14)
    X = rng.standard_normal((20000, 20)).astype(dtype)
    Q = rng.standard_normal((6100, 20)).astype(dtype)
    odd = [3, 4, 5, 6099]
    Q[3, 1], Q[4, 0], Q[5, 19], Q[6099] = np.nan, np.inf, -np.inf, np.nan
    nfb = _compare(X, Q, 5, most_listed=600)
    assert nfb >= len(odd)
    X[77, 3], X[78, 0], X[19999, 19] = np.nan, np.inf, -np.inf
    nn = aoclda.neighbors.nearest_neighbors().fit(X)
    tile = aoclda.neighbors.nearest_neighbors(seed_thresholds=False).fit(X)
    for part in (Q, np.delete(Q, odd, axis=0)):
        dist, ind = nn.kneighbors(part, n_neighbors=5)
        assert _stats(nn)[1] != KEEP
        de, ie = tile.kneighbors(part, n_neighbors=5)
        np.testing.assert_array_equal(ind, ie)
        np.testing.assert_array_equal(dist, de)
    assert not np.isin(ind, [77, 78, 19999]).any()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,d,k", [(20011, 20, 10), (16385, 64, 100), (66000, 100, 1),
                                   (140000, 16, 20), (8192, 128, 128)])
def test_ordinary_data_against_the_oracle(oracle, dtype, n, d, k):
    """Fewer than one query in ten is left to the tile, and none comes out differently: all by the
    tile, and the first 150 by the oracle."""
    rng = np.random.default_rng(n + d)
    means = rng.uniform(-10, 10, (16, d))
    X = _mixture(rng, n, d, dtype, means)
    Q = _mixture(rng, _queries(n, d), d, dtype, means)
    _compare(X, Q, k, most_listed=len(Q) // 10)
    dist, ind = aoclda.neighbors.nearest_neighbors().fit(X).kneighbors(Q, n_neighbors=k)
    ei, ed = oracle.knn(X.astype(np.float64), Q[:150].astype(np.float64), k)
    np.testing.assert_array_equal(ind[:150], ei)
    np.testing.assert_allclose(dist[:150], ed, rtol=1e-14 if dtype == np.float64 else 1.2e-7)
