"""IVF-Flat search by matrix-core scores against the list scans, which serve k > 128: the scans'
first k neighbours of a k = 129 search are the answer, bit for bit (both sum and round exact keys
alike, ties by list and position)."""
import ctypes as C

import numpy as np
import pytest

import aoclda
from aoclda import _lib as L

pytestmark = pytest.mark.gpu


def _check(ann, Q, ks, k_scan=129):
    de, ie = ann.kneighbors(Q, n_neighbors=k_scan)
    for k in ks:
        dist, ind = ann.kneighbors(Q, n_neighbors=k)
        np.testing.assert_array_equal(ind, ie[:, :k], err_msg=f"k {k}")
        np.testing.assert_array_equal(dist, de[:, :k], err_msg=f"k {k}")


@pytest.mark.parametrize("metric", ["sqeuclidean", "euclidean", "inner product", "cosine"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", [1, 31, 32, 33, 64, 65, 96, 97, 127, 128])
def test_same_as_scan(metric, dtype, d):
    """One to four k steps and their edges; lists of one to several runs of tiles."""
    rng = np.random.default_rng(d)
    means = rng.uniform(-3, 3, (12, d))
    X = (means[rng.integers(0, 12, 5003)] + rng.standard_normal((5003, d))).astype(dtype)
    Q = (means[rng.integers(0, 12, 333)] + rng.standard_normal((333, d))).astype(dtype)
    ann = aoclda.neighbors.approximate_neighbors(n_list=17, n_probe=5, metric=metric,
                                                 kmeans_iter=3, seed=1).train_and_add(X)
    _check(ann, Q, (1, 10, 128))


@pytest.mark.parametrize("nq", [1, 15, 16, 17, 128, 129, 700])
@pytest.mark.parametrize("n,n_list,n_probe", [(300, 200, 200), (300, 200, 3), (4096, 1, 1),
                                              (9000, 3, 2)])
def test_groups(nq, n, n_list, n_probe):
    """Groups of one to several hundred queries; lists shorter than a tile, empty, longer than a
    run; fewer vectors than k in the probed lists (index -1)."""
    rng = np.random.default_rng(nq)
    X = rng.standard_normal((n, 20)).astype(np.float32)
    Q = rng.standard_normal((nq, 20)).astype(np.float32)
    ann = aoclda.neighbors.approximate_neighbors(n_list=n_list, n_probe=n_probe, kmeans_iter=2,
                                                 seed=1).train_and_add(X)
    _check(ann, Q, (1, 33, 128))


@pytest.mark.parametrize("metric", ["sqeuclidean", "inner product"])
def test_ties_and_added_copies(metric):
    """Equal keys keep list and position order: integer rows, each added three times, so that up
    to hundreds of keys tie; more than 1,024 equal rows go to the scan."""
    rng = np.random.default_rng(5)
    X = rng.integers(0, 3, (2000, 6)).astype(np.float32)
    ann = aoclda.neighbors.approximate_neighbors(n_list=8, n_probe=4, metric=metric, kmeans_iter=3,
                                                 seed=2).train_and_add(X)
    Q = rng.integers(0, 3, (90, 6)).astype(np.float32)
    _check(ann, Q, (1, 50, 128))
    ann.add(X)
    ann.add(np.repeat(X[:1], 1500, axis=0))
    _check(ann, np.concatenate([Q, X[:1]]), (1, 50, 128))


@pytest.mark.parametrize("dtype,scale", [(np.float32, 1e-25), (np.float32, 1e18),
                                         (np.float64, 1e-150), (np.float64, 1e70),
                                         (np.float32, 1e-3)])
@pytest.mark.parametrize("metric", ["sqeuclidean", "inner product"])
def test_ranges(dtype, scale, metric):
    """Keys that round to zero or overflow in the type, and queries far outside the data's range
    beside ordinary ones."""
    rng = np.random.default_rng(9)
    X = (rng.standard_normal((3000, 24)) * scale).astype(dtype)
    Q = (rng.standard_normal((40, 24)) * scale).astype(dtype)
    Q[3] *= dtype(100)
    Q[7] *= dtype(1e-6)
    Q[11] = 0
    ann = aoclda.neighbors.approximate_neighbors(n_list=10, n_probe=4, metric=metric, kmeans_iter=2,
                                                 seed=1).train_and_add(X)
    _check(ann, Q, (1, 10, 128))


def _launches(ann):
    """Launches of (list-major scores, scans) since the last call."""
    out = []
    for name in (b"ivf_tile_scores", b"ivf_scan"):
        ms, cnt = C.c_double(), L.da_int()
        st = L.lib.da_amd_profile_get(ann._h.h, name, C.byref(ms), C.byref(cnt))
        out.append(cnt.value if st == 0 else 0)
    L.check(L.lib.da_amd_profile_reset(ann._h.h))
    return tuple(out)


@pytest.mark.parametrize("metric", ["sqeuclidean", "euclidean", "inner product", "cosine"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", [1, 20, 33, 128])
def test_served_by_the_tiles(metric, dtype, d):
    """Ordinary data are searched by the matrix-core scores alone; only a query with more than 1,024
    equal vectors takes the scan beside them."""
    rng = np.random.default_rng(d)
    X = rng.standard_normal((6000, d)).astype(dtype)
    Q = rng.standard_normal((300, d)).astype(dtype)
    if d == 1:
        X, Q = X * dtype(30) + dtype(100), Q * dtype(30) + dtype(100)
    ann = aoclda.neighbors.approximate_neighbors(n_list=12, n_probe=4, metric=metric,
                                                 kmeans_iter=3, seed=1).train_and_add(X)
    L.check(L.lib.da_amd_profile_enable(ann._h.h, 1))
    _check(ann, Q, ())
    assert _launches(ann) == (0, 1)  # k = 129
    for k in (1, 10, 128):
        ann.kneighbors(Q, n_neighbors=k)
        if d > 1 or metric != "cosine":  # every cosine of one feature is 1
            assert _launches(ann) == (1, 0)
        else:
            assert _launches(ann)[0] == 1
    if metric != "inner product":
        ann.add(np.repeat(X[:1], 1500, axis=0))
        _check(ann, X[:40], (5,))
        assert _launches(ann) == (1, 2)


def test_layout_after_a_change():
    """A few queries after a change of the index are scanned; a second search, or a first one that
    scans eight times the index and 2^20 vectors, lays the lists out."""
    rng = np.random.default_rng(3)
    X = rng.standard_normal((140000, 24)).astype(np.float32)
    Q = rng.standard_normal((4000, 24)).astype(np.float32)
    ann = aoclda.neighbors.approximate_neighbors(n_neighbors=7, n_list=40, n_probe=4,
                                                 kmeans_iter=3, seed=1).train_and_add(X)
    L.check(L.lib.da_amd_profile_enable(ann._h.h, 1))
    want = ann.kneighbors(Q, n_neighbors=129)  # counts as the first search
    assert _launches(ann) == (0, 1)

    def search(nq):
        dist, ind = ann.kneighbors(Q[:nq])
        np.testing.assert_array_equal(ind, want[1][:nq, :7])
        np.testing.assert_array_equal(dist, want[0][:nq, :7])
        return _launches(ann)

    assert search(5) == (1, 0)
    far = np.full((1, 24), 50, np.float32)  # in nobody's neighbourhood
    ann.add(far)
    assert [search(79), search(5), search(4000)] == [(0, 1), (1, 0), (1, 0)]
    ann.add(far)
    assert search(80) == (1, 0)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,d,n_list,n_probe,nq,k,small", [
    (2000, 8, 64, 1, 1, 10, True), (2000, 8, 64, 1, 1000, 10, True), (2000, 8, 64, 4, 1000, 10, False),
    (1200, 32, 26, 20, 7, 88, True), (4096, 20, 1, 1, 1, 1, False), (600, 80, 98, 44, 1, 2, True),
    (10000, 120, 64, 4, 64, 10, False), (12, 3, 1, 1, 1, 1, True)])
def test_small_searches(dtype, n, d, n_list, n_probe, nq, k, small):
    """Small searches are scanned however often they are made, and leave no layout behind; the same
    answers on either side of the line."""
    rng = np.random.default_rng(n)
    X, Q = rng.standard_normal((n, d)).astype(dtype), rng.standard_normal((nq, d)).astype(dtype)
    ann = aoclda.neighbors.approximate_neighbors(n_list=n_list, n_probe=n_probe, kmeans_iter=2,
                                                 seed=1).train_and_add(X)
    L.check(L.lib.da_amd_profile_enable(ann._h.h, 1))
    for i in range(3):
        dist, ind = ann.kneighbors(Q, n_neighbors=k)
    assert _launches(ann)[0] == (0 if small else 2)
    if n > 129:
        de, ie = ann.kneighbors(Q, n_neighbors=129)
        np.testing.assert_array_equal(ind, ie[:, :k])
        np.testing.assert_array_equal(dist, de[:, :k])


@pytest.mark.parametrize("metric", ["sqeuclidean", "inner product", "cosine"])
@pytest.mark.parametrize("where", ["rows", "queries"])
def test_not_finite(metric, where):
    """Vectors that are not finite leave the index to the scans, such queries themselves."""
    rng = np.random.default_rng(6)
    X = rng.standard_normal((5000, 24)).astype(np.float32)
    Q = rng.standard_normal((60, 24)).astype(np.float32)
    ann = aoclda.neighbors.approximate_neighbors(n_list=10, n_probe=4, metric=metric, kmeans_iter=2,
                                                 seed=1).train_and_add(X)
    L.check(L.lib.da_amd_profile_enable(ann._h.h, 1))
    if where == "rows":
        bad = X[:3].copy()
        bad[0, 3], bad[1, 0], bad[2, 5] = np.nan, np.inf, -np.inf
        ann.add(bad)
    else:
        Q[7, 3], Q[8, 0], Q[9, 5], Q[10] = np.nan, np.inf, -np.inf, 3e37
    _launches(ann)
    with np.errstate(all="ignore"):
        _check(ann, Q, (1, 10, 128))
    tiles, scans = _launches(ann)
    assert (tiles, scans) == ((0, 4) if where == "rows" else (3, 4))
