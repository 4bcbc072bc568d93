"""Radius search and DBSCAN of the squared-euclidean metrics, up to 128 features: small searches,
which take key tiles, against the oracle; large ones (2,048 queries and 2^28 pairs, DBSCAN of 4,096
rows), which go through the matrix-core hit bits, against the oracle and against key tiles: tile
edges, padded widths, rows that need the exact re-check, and the data that send the search to the
general path."""
import ctypes as C

import numpy as np
import pytest

import aoclda
from aoclda import _lib as L

pytestmark = pytest.mark.gpu


def blobs(rng, n, d, dtype, sigma=0.5, offset=0.0):
    means = rng.uniform(-10, 10, (8, d)) + offset
    return (means[rng.integers(0, 8, n)] + sigma * rng.standard_normal((n, d))).astype(dtype)


def radius_of(X, Q, share):
    """A radius that keeps about this share of the training rows."""
    s = np.sqrt(((X[None, :400].astype(np.float64) - Q[:50, None].astype(np.float64)) ** 2).sum(-1))
    return float(np.quantile(s, share))


# Edges: 64-row words, 128- and 256-row blocks, every k-step count, the smallest width.
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,nq,d", [(2048, 2048, 1), (2049, 2050, 3), (2111, 2300, 16),
                                    (2113, 2047, 32), (2500, 1700, 33), (3000, 1500, 65),
                                    (2100, 2100, 97), (2304, 1900, 128)])
@pytest.mark.parametrize("metric", ["euclidean", "sqeuclidean", "euclidean_gemm"])
def test_radius(oracle, dtype, n, nq, d, metric):
    rng = np.random.default_rng(n + d)
    X, Q = blobs(rng, n, d, dtype), blobs(rng, nq, d, dtype)
    Q[:7] = X[:7]
    r = radius_of(X, Q, 0.03)
    r = float(dtype(r * r if metric == "sqeuclidean" else r))
    nn = aoclda.neighbors.nearest_neighbors(metric=metric, radius=r).fit(X)
    dist, ind = nn.radius_neighbors(Q)
    cnt, ei, ed = oracle.radius(X, Q, r, metric, single=dtype == np.float32)
    # The GEMM-form metric may differ where the key equals the threshold up to its rounding
    # (absolute, about 1e-12 of the squared norms); none of these data has such a pair.
    assert [len(v) for v in ind] == list(cnt)
    np.testing.assert_array_equal(np.concatenate(list(ind)), ei)
    # fp32: one rounding (2^-24). The GEMM form's squared key |x|^2 + |y|^2 - 2 x.y is off by up
    # to 2 (d + 2) 2^-53 (|x|^2 + |y|^2), its root by up to the root of that (at distance 0).
    tol = 1e-6 if dtype == np.float32 else 1e-12
    big = max((X.astype(np.float64) ** 2).sum(1).max(), (Q.astype(np.float64) ** 2).sum(1).max())
    atol = np.sqrt(2 * (d + 2) * 2.0 ** -53 * 2 * big) if metric == "euclidean_gemm" else tol
    np.testing.assert_allclose(np.concatenate(list(dist)), ed, rtol=tol, atol=atol)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", ["offset", "duplicates", "all", "outlier", "boundary", "tiny",
                                  "nonfinite"])
def test_dbscan_data(oracle, dtype, case):
    """Data far from the origin, exact duplicates with eps = 0, every pair a neighbour, an
    outlier that makes every pair of a blob borderline, distances equal to eps, subnormal scales,
    and values that are not finite."""
    rng = np.random.default_rng(5)
    n, d, eps = 2300, 6, 0.9
    X = blobs(rng, n, d, dtype)
    if case == "offset":
        X = blobs(rng, n, d, dtype, offset=3e4 if dtype == np.float32 else 1e8)
    elif case == "duplicates":
        X, eps = X[rng.integers(0, 300, n)], 0.0
    elif case == "all":
        eps = 1e4
    elif case == "outlier":
        X[17] = 1e9
    elif case == "boundary":
        X = rng.integers(0, 12, (n, d)).astype(dtype)
        eps = 3.0  # integer squared distances: many equal 9
    elif case == "tiny":
        scale = dtype(1e-18 if dtype == np.float32 else 1e-140)
        X, eps = X * scale, float(dtype(0.9) * scale)
    elif case == "nonfinite":
        X[3, 2], X[100, 0], X[101, 5] = np.nan, np.inf, -np.inf
    db = aoclda.clustering.DBSCAN(eps=eps, min_samples=6, algorithm="brute").fit(X)
    with np.errstate(all="ignore"):
        labels, core, nc = oracle.dbscan(X, eps, 6, single=dtype == np.float32)
    np.testing.assert_array_equal(db.labels, labels)
    np.testing.assert_array_equal(db.core_sample_indices, np.flatnonzero(core))
    assert db.n_clusters == nc


@pytest.mark.parametrize("metric", ["euclidean", "l2", "sqeuclidean"])
@pytest.mark.parametrize("d", [2, 40, 128])
def test_dbscan_metrics(oracle, metric, d):
    rng = np.random.default_rng(d)
    X = blobs(rng, 2600, d, np.float32)
    eps = radius_of(X, X, 0.02)
    eps = float(np.float32(eps * eps if metric == "sqeuclidean" else eps))
    db = aoclda.clustering.DBSCAN(eps=eps, min_samples=5, metric=metric, algorithm="brute").fit(X)
    labels, core, _ = oracle.dbscan(X, eps, 5, metric, single=True)
    np.testing.assert_array_equal(db.labels, labels)
    np.testing.assert_array_equal(db.core_sample_indices, np.flatnonzero(core))


def test_dbscan_several_blocks():
    """Several blocks of bits and a ragged last one: core samples and clusters against a k-d tree."""
    from scipy.sparse import coo_matrix
    from scipy.sparse.csgraph import connected_components
    from scipy.spatial import cKDTree
    rng = np.random.default_rng(23)
    means = rng.uniform(-50, 50, (300, 3))
    X = means[rng.integers(0, 300, 140001)] + rng.standard_normal((140001, 3))
    eps, min_samples = 0.3, 8
    db = aoclda.clustering.DBSCAN(eps=eps, min_samples=min_samples).fit(X)
    tree = cKDTree(X)
    pairs = tree.query_pairs(eps, output_type="ndarray")
    deg = np.bincount(pairs.ravel(), minlength=len(X)) + 1
    core = deg >= min_samples
    np.testing.assert_array_equal(np.sort(np.asarray(db.core_sample_indices)), np.flatnonzero(core))
    cc = pairs[core[pairs[:, 0]] & core[pairs[:, 1]]]
    g = coo_matrix((np.ones(len(cc)), (cc[:, 0], cc[:, 1])), shape=(len(X), len(X)))
    _, comp = connected_components(g, directed=False)
    lab = np.asarray(db.labels)
    first = {}
    for c, l in zip(comp[core], lab[core]):
        assert first.setdefault(c, l) == l
    assert len(set(first.values())) == len(first) == db.n_clusters


def _sliced(nn, Q, step=60, **kw):
    """The search a few queries at a time, which takes the key tiles of the general path."""
    parts = [nn.radius_neighbors(Q[i:i + step], **kw) for i in range(0, len(Q), step)]
    return [np.concatenate([np.concatenate([[], *v]) for v in p]) for p in
            (zip(*parts) if isinstance(parts[0], tuple) else [parts])]


class _Profiled(L.Handle):
    def __init__(self, *args):
        super().__init__(*args)
        L.check(L.lib.da_amd_profile_enable(self.h, 1))


@pytest.fixture
def profiled(monkeypatch):
    """Handles count their kernels: launches(handle, name)."""
    monkeypatch.setattr(L, "Handle", _Profiled)

    def launches(handle, name):
        ms, cnt = C.c_double(), L.da_int()
        st = L.lib.da_amd_profile_get(handle.h, name.encode(), C.byref(ms), C.byref(cnt))
        return cnt.value if st == 0 else 0

    return launches


def _same(nn, Q, profiled, step, served=True, **kw):
    """The whole search, bit for bit that of the slices; by hit bits from end to end (served)."""
    L.check(L.lib.da_amd_profile_reset(nn._h.h))
    got = nn.radius_neighbors(Q, **kw)
    n_verify, n_fill = profiled(nn._h, "radius_verify"), profiled(nn._h, "pairwise_direct")
    assert (n_verify > 0 and n_fill == 0) == served
    parts = got if isinstance(got, tuple) else [got]
    for a, b in zip(parts, _sliced(nn, Q, step, **kw)):
        np.testing.assert_array_equal(np.concatenate(list(a)), b)
    assert profiled(nn._h, "radius_verify") == n_verify  # the slices went another way
    return got


# Every k-step count and the smallest width; edges of 512-row blocks and of 128- and 256-row blocks.
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,nq,d", [(65536, 4096, 1), (65537, 4098, 3), (66111, 4300, 16),
                                    (65600, 4223, 32), (66000, 4097, 33), (131073, 2048, 65),
                                    (65537, 4400, 97), (66048, 4352, 128)])
@pytest.mark.parametrize("metric", ["euclidean", "sqeuclidean", "euclidean_gemm"])
def test_radius_hit_bits(profiled, dtype, n, nq, d, metric):
    rng = np.random.default_rng(n + d)
    X, Q = blobs(rng, n, d, dtype), blobs(rng, nq, d, dtype)
    Q[:7] = X[:7]
    r = radius_of(X, Q, 0.002)
    r = float(dtype(r * r if metric == "sqeuclidean" else r))
    nn = aoclda.neighbors.nearest_neighbors(metric=metric, radius=r).fit(X)
    _same(nn, Q, profiled, 1000)


def test_radius_blocks_and_switch(profiled):
    """Several blocks of queries and a ragged last one; the same with a run of queries in the
    second block that hold so many rows that the rest of the search takes key tiles, though the
    rows looked at before the sweep do not show it."""
    rng = np.random.default_rng(8)
    X = rng.uniform(-10, 10, (65536, 3)).astype(np.float32)
    X[:32768] = 0.1 * rng.standard_normal((32768, 3)) + 20
    Q = rng.uniform(-10, 10, (33003, 3)).astype(np.float32)
    nn = aoclda.neighbors.nearest_neighbors(radius=0.5).fit(X)
    _same(nn, Q, profiled, 1500, return_distance=False)
    _same(nn, Q[:20000], profiled, 1500, sort_results=True)
    Q[17000:20500] = 0.1 * rng.standard_normal((3500, 3)) + 20
    nn = aoclda.neighbors.nearest_neighbors(radius=0.5).fit(X)
    _same(nn, Q, profiled, 1500, served=False, return_distance=False)
    assert profiled(nn._h, "radius_verify") == 1


@pytest.mark.parametrize("case", ["outlier", "nonfinite", "dense"])
def test_radius_general_path(profiled, case):
    """Large searches whose data the bits cannot separate, hold values that are not finite, or
    whose radius holds too many rows."""
    rng = np.random.default_rng(9)
    X, Q = blobs(rng, 65536, 6, np.float32), blobs(rng, 4100, 6, np.float32)
    r = radius_of(X, Q, 0.05 if case == "dense" else 0.002)
    if case == "outlier":
        X[17] = 1e9
    elif case == "nonfinite":
        X[3, 2], X[100, 0], Q[11, 5] = np.nan, np.inf, -np.inf
    nn = aoclda.neighbors.nearest_neighbors(radius=r).fit(X)
    _same(nn, Q, profiled, 1000, served=False, return_distance=False)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,d,metric", [(4096, 1, "euclidean"), (4097, 3, "l2"),
                                        (4159, 16, "sqeuclidean"), (4161, 32, "euclidean"),
                                        (4607, 33, "l2"), (4609, 65, "sqeuclidean"),
                                        (5000, 97, "euclidean"), (4224, 128, "l2")])
def test_dbscan_hit_bits(oracle, profiled, dtype, n, d, metric):
    rng = np.random.default_rng(n)
    X = blobs(rng, n, d, dtype)
    eps = radius_of(X, X, 0.004)
    eps = float(dtype(eps * eps if metric == "sqeuclidean" else eps))
    db = aoclda.clustering.DBSCAN(eps=eps, min_samples=5, metric=metric, algorithm="brute").fit(X)
    assert profiled(db._h, "radius_verify") == 1 and profiled(db._h, "pairwise_direct") == 0
    labels, core, nc = oracle.dbscan(X, eps, 5, metric, single=dtype == np.float32)
    np.testing.assert_array_equal(db.labels, labels)
    np.testing.assert_array_equal(db.core_sample_indices, np.flatnonzero(core))
    assert db.n_clusters == nc


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", ["offset", "duplicates", "all", "outlier", "boundary",
                                  "nonfinite", "hidden"])
def test_dbscan_hit_bits_data(oracle, profiled, dtype, case):
    """As test_dbscan_data, at a size of the hit bits; "hidden": more hits than the rows looked at
    before the sweep show."""
    rng = np.random.default_rng(5)
    n, d, eps, served = 4300, 6, 0.6, True
    X = blobs(rng, n, d, dtype)
    if case == "offset":
        X = blobs(rng, n, d, dtype, offset=3e4 if dtype == np.float32 else 1e8)
    elif case == "duplicates":
        X, eps = X[rng.integers(0, 500, n)], 0.0
    elif case == "all":
        eps, served = 1e4, False
    elif case == "outlier":
        X[17], served = 1e9, False
    elif case == "boundary":
        X, eps = rng.integers(0, 40, (n, d)).astype(dtype), 9.0  # many squared distances equal 81
    elif case == "nonfinite":
        X[3, 2], X[100, 0], X[101, 5], served = np.nan, np.inf, -np.inf, False
    elif case == "hidden":
        X[256:1000] = 1e-3 * rng.standard_normal((744, d))
        X[1300:2000] = 1e-3 * rng.standard_normal((700, d))
        served = False
    db = aoclda.clustering.DBSCAN(eps=eps, min_samples=6, algorithm="brute").fit(X)
    assert (profiled(db._h, "radius_verify") > 0) == served
    with np.errstate(all="ignore"):
        labels, core, nc = oracle.dbscan(X, eps, 6, single=dtype == np.float32)
    np.testing.assert_array_equal(db.labels, labels)
    np.testing.assert_array_equal(db.core_sample_indices, np.flatnonzero(core))
    assert db.n_clusters == nc


# 1e-20 to 3e-22: squared distances about float's smallest normal number and below it; 1e-23: the
# squared radius is 0 in float, and so is the key of every pair within a few of its units.
SMALL = [1e-20, 1e-21, 3e-22, 1e-22, 5e-23, 1e-23, 1e-25]


@pytest.mark.parametrize("scale", SMALL)
@pytest.mark.parametrize("metric", ["euclidean", "sqeuclidean", "euclidean_gemm"])
def test_radius_below_the_normal_range(oracle, scale, metric):
    """Keys are rounded to float before they are compared; below its normal range by an absolute
    amount that lets pairs beyond the radius in. Against key tiles, and for a few queries against
    the oracle."""
    X = (blobs(np.random.default_rng(31), 66000, 6, np.float64) * scale).astype(np.float32)
    Q = (blobs(np.random.default_rng(31), 4100, 6, np.float64) * scale).astype(np.float32)
    r = np.float32(0.5 * scale)
    r = float(r * r if metric == "sqeuclidean" else r)
    nn = aoclda.neighbors.nearest_neighbors(metric=metric, radius=r).fit(X)
    ind = nn.radius_neighbors(Q, return_distance=False)
    cnt, ei, _ = oracle.radius(X, Q[:60], r, metric, single=True)
    np.testing.assert_array_equal([len(v) for v in ind[:60]], cnt)
    np.testing.assert_array_equal(np.concatenate(list(ind[:60])), ei)
    np.testing.assert_array_equal(np.concatenate(list(ind)),
                                  _sliced(nn, Q, 1000, return_distance=False)[0])


@pytest.mark.parametrize("scale", SMALL + [1e-30, 1e-43])
@pytest.mark.parametrize("metric", ["euclidean", "l2", "sqeuclidean"])
def test_dbscan_below_the_normal_range(oracle, scale, metric):
    rng = np.random.default_rng(32)
    X = (blobs(rng, 4200, 6, np.float64) * scale).astype(np.float32)
    eps = np.float32(0.6 * scale)
    eps = float(eps * eps if metric == "sqeuclidean" else eps)
    db = aoclda.clustering.DBSCAN(eps=eps, min_samples=6, metric=metric, algorithm="brute").fit(X)
    labels, core, _ = oracle.dbscan(X, eps, 6, metric, single=True)
    np.testing.assert_array_equal(db.labels, labels)
    np.testing.assert_array_equal(db.core_sample_indices, np.flatnonzero(core))
