"""k-means++ on the device: every width of its row stage (rows of up to 4, 8 and 16 16-byte pieces a
thread, and wider or unaligned ones), every slot count of the candidates (k below 403 and above),
several starts, the spherical form and data whose rows all coincide, against the oracle's draws."""
import numpy as np
import pytest

import aoclda

pytestmark = pytest.mark.gpu


def _blobs(seed, n, d, k, dtype, spread=0.3):
    rng = np.random.default_rng(seed)
    means = rng.uniform(-10, 10, (k, d))
    return (means[rng.integers(0, k, n)] + spread * rng.standard_normal((n, d))).astype(dtype)


def _check(oracle, X, k, dtype, n_init=1, max_iter=6):
    km = aoclda.clustering.kmeans(n_clusters=k, initialization_method="k-means++", n_init=n_init,
                                  seed=17, max_iter=max_iter, tol=0.0).fit(X)
    r = oracle.kmeans(X.astype(np.float64), k, "k-means++", n_init=n_init, seed=17,
                      max_iter=max_iter, tol=0.0)
    np.testing.assert_array_equal(km.labels, r["labels"])
    # The centres are double means of the same rows, reported in the data's precision.
    rtol = 1e-12 if dtype == np.float64 else 1e-5
    np.testing.assert_allclose(km.cluster_centres, r["centres"], rtol=rtol, atol=rtol)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("d", [1, 2, 3, 4, 7, 8, 15, 16, 17, 31, 32, 33, 64, 65, 130])
def test_row_widths(oracle, dtype, d):
    _check(oracle, _blobs(d, 1037, d, 9, dtype), 9, dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("d", [79, 80, 81, 96, 97, 127, 128, 129, 600])
def test_wide_rows(oracle, dtype, d):
    """Rows staged 16 or 32 features at a time, the next ones read ahead: whole and partial stages,
    a last step of a few rows."""
    _check(oracle, _blobs(d, 773, d, 5, dtype), 5, dtype, max_iter=2)


@pytest.mark.parametrize("n", [2, 255, 256, 257, 2048, 2049, 20001])
def test_row_counts(oracle, n):
    k = 2 if n == 2 else 6
    _check(oracle, _blobs(n, n, 5, k, np.float32), k, np.float32)


@pytest.mark.parametrize("k", [2, 3, 7, 8, 54, 55, 402, 404, 1100])
def test_candidate_slots(oracle, k):
    """2 + log(k) candidates: 2 to 9, with the last centre 3 to 10 slots of 4, 8 and 16. (Two
    candidates of a round that are each other's nearest sample cost exactly the same, and the
    rounding of the sums decides; with 5 rows a centre or more no round of these data has a pair.)"""
    n = 1300 if k < 100 else 6000
    _check(oracle, _blobs(k, n, 6, 40, np.float64, 1.0), k, np.float64, max_iter=2)


def test_several_starts(oracle):
    _check(oracle, _blobs(5, 900, 6, 12, np.float64), 12, np.float64, n_init=5)


def test_coinciding_rows():
    """Every row the same: the first k rows are taken and no draw is made."""
    X = np.full((300, 5), 2.5, np.float32)
    km = aoclda.clustering.kmeans(n_clusters=3, initialization_method="k-means++", n_init=1, seed=3,
                                  max_iter=3, tol=0.0).fit(X)
    np.testing.assert_array_equal(km.labels, np.zeros(300, np.int32))
    assert km.inertia == 0


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_spherical(oracle, dtype):
    X = _blobs(8, 1500, 12, 7, dtype)
    km = aoclda.clustering.kmeans(n_clusters=7, n_init=1, seed=3, max_iter=5, tol=1e-8,
                                  distance="cosine", normalize_data=True).fit(X)
    r = oracle.kmeans_sph(X.astype(np.float64), 7, "k-means++", n_init=1, seed=3, max_iter=5,
                          tol=1e-8, normalize=True)
    np.testing.assert_array_equal(km.labels, r["labels"])
