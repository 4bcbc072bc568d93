"""Batched k-means at the edges of its chunks: instances of a few rows, of one row more or less than a
tile or a chunk, rows that start off the 16-byte boundary, and one that is not finite beside others."""
import numpy as np
import pytest

import aoclda

pytestmark = pytest.mark.gpu


def _instance(rng, n, d, k):
    means = rng.uniform(-10, 10, (k, d))
    X = (means[rng.integers(0, k, n)] + rng.standard_normal((n, d))).astype(np.float32)
    return X, X[:k].copy()


def _check(oracle, data, inits, out, skip=()):
    cs, labs, n_iter, inertia = out
    for i, X in enumerate(data):
        if i in skip:
            continue
        r = oracle.kmeans(X.astype(np.float64), len(inits[i]), "supplied",
                          inits[i].astype(np.float64), max_iter=8, tol=0.0)
        np.testing.assert_array_equal(labs[i], r["labels"], err_msg=f"instance {i} {X.shape}")
        assert n_iter[i] == r["n_iter"]
        # Double means and sums reported in fp32.
        np.testing.assert_allclose(cs[i], r["centres"], rtol=1e-5, atol=1e-5)
        np.testing.assert_allclose(inertia[i], r["inertia"], rtol=1e-5)


@pytest.mark.parametrize("d", [1, 3, 5, 16, 17, 63, 64])
def test_sizes(oracle, d):
    rng = np.random.default_rng(d)
    data, inits = [], []
    for n in (2, 3, 15, 16, 17, 63, 64, 65, 255, 257, 511, 513, 1023, 1025, 2047, 2049, 4099, 20001):
        X, C = _instance(rng, n, d, 2 if n < 64 else 7)
        data.append(X)
        inits.append(C)
    _check(oracle, data, inits, aoclda.clustering.kmeans_batch(data, inits, 8, 0.0, "working"))


def test_one_instance_not_finite(oracle):
    rng = np.random.default_rng(3)
    data, inits = zip(*[_instance(rng, n, 6, 4) for n in (700, 900, 1100)])
    data, inits = list(data), list(inits)
    data[1][500, 2] = np.inf
    _check(oracle, data, inits, aoclda.clustering.kmeans_batch(data, inits, 8, 0.0, "working"),
           skip=(1,))
