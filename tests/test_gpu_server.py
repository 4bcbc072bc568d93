"""Serving loop (da_nn_server_*): continuous batching must not change any result. Each
request's neighbours are compared alone, mixed with others, and against the oracle."""
import ctypes as C

import numpy as np
import pytest

import aoclda
from aoclda import _lib as L
from aoclda.neighbors import nn_server

pytestmark = pytest.mark.gpu


def unit_rows(rng, n, means, sigma=0.1):
    comp = rng.integers(0, len(means), n)
    X = means[comp] + sigma * rng.standard_normal((n, means.shape[1]))
    return X / np.linalg.norm(X, axis=1, keepdims=True)


@pytest.mark.parametrize("precision", ["working", "fp16", "bf16"])
def test_alone_equals_mixed(oracle, precision):
    rng = np.random.default_rng(31)
    means = rng.standard_normal((64, 96))
    Xt = unit_rows(rng, 20000, means).astype(np.float32)
    nn = aoclda.neighbors.nearest_neighbors(precision=precision).fit(Xt)
    sizes = [1, 3, 17, 250, 700, 2049, 5]
    ks = [1, 10, 16, 10, 1, 16, 10]
    reqs = [unit_rows(rng, s, means).astype(np.float32) for s in sizes]
    srv = nn_server(nn, max_batch_queries=1024, max_device_bytes=64 << 20)
    alone = []
    for X, k in zip(reqs, ks):
        rid = srv.submit(X, k)
        alone.append(srv.wait(rid))
    ids = [srv.submit(X, k) for X, k in zip(reqs, ks)]
    mixed = [srv.wait(r) for r in ids]
    for (da, ia, la), (dm, im, lm), X, k in zip(alone, mixed, reqs, ks):
        np.testing.assert_array_equal(ia, im)
        np.testing.assert_array_equal(da, dm)
        ei, ed = oracle.knn(Xt.astype(np.float64), X.astype(np.float64), k)
        np.testing.assert_array_equal(ia, ei)
        np.testing.assert_allclose(da, ed, rtol=1e-5, atol=1e-6)
        assert la > 0 and lm > 0
    st = srv.stats()
    assert st["requests"] == 2 * len(sizes)
    assert st["queries"] == 2 * sum(sizes)
    # the 2049-query request exceeds a 1024-query batch and is served in slices
    assert st["batches"] >= 4
    srv.close()


def test_argument_errors():
    rng = np.random.default_rng(32)
    Xt = rng.standard_normal((100, 8)).astype(np.float32)
    nn = aoclda.neighbors.nearest_neighbors().fit(Xt)
    srv = nn_server(nn, max_batch_queries=64)
    with pytest.raises(aoclda.DAError):
        srv.submit(np.ones((2, 7), dtype=np.float32), 3)  # wrong feature count
    with pytest.raises(aoclda.DAError):
        srv.submit(np.ones((2, 8), dtype=np.float32), 101)  # k > n_samples
    srv.close()


@pytest.mark.parametrize("precision,dtype", [("fp16x3", np.float32), ("bf16x3", np.float32),
                                             ("working", np.float64)])
def test_mixed_k_and_short_lists(oracle, precision, dtype):
    """Requests with k above 32 (candidate lists shorter than k, the batch searched at its
    largest k and the smaller requests taking a prefix) submitted together with k = 1 and
    k = 50: every result equals the request served alone and the oracle, also for the split
    16-bit forms and an fp64 server."""
    rng = np.random.default_rng(33)
    means = rng.standard_normal((64, 48))
    Xt = unit_rows(rng, 30000, means).astype(dtype)
    nn = aoclda.neighbors.nearest_neighbors(precision=precision).fit(Xt)
    sizes = [40, 7, 300, 129, 1]
    ks = [33, 128, 50, 1, 100]
    reqs = [unit_rows(rng, s, means).astype(dtype) for s in sizes]
    srv = nn_server(nn, max_batch_queries=256, max_device_bytes=64 << 20)
    alone = [srv.wait(srv.submit(X, k)) for X, k in zip(reqs, ks)]
    ids = [srv.submit(X, k) for X, k in zip(reqs, ks)]
    mixed = [srv.wait(r) for r in ids]
    rtol = 1e-12 if dtype == np.float64 else 1e-5
    for (da, ia, _), (dm, im, _), X, k in zip(alone, mixed, reqs, ks):
        np.testing.assert_array_equal(ia, im)
        np.testing.assert_array_equal(da, dm)
        ei, ed = oracle.knn(Xt.astype(np.float64), X.astype(np.float64), k)
        np.testing.assert_array_equal(ia, ei)
        np.testing.assert_allclose(da, ed, rtol=rtol, atol=1e-6 if dtype == np.float32 else 0)
    srv.close()


def test_second_wait_on_a_request_is_refused():
    """A result goes to one waiter: waiting again on a finished request, or from a second
    thread while the first still waits, returns invalid_input instead of touching freed
    state."""
    import threading
    rng = np.random.default_rng(34)
    Xt = rng.standard_normal((5000, 16)).astype(np.float32)
    nn = aoclda.neighbors.nearest_neighbors().fit(Xt)
    srv = nn_server(nn, max_batch_queries=64)
    rid = srv.submit(Xt[:500], 10)
    nq, k = srv._k[rid]
    results = []

    def waiter():
        ind = np.empty((nq, k), dtype=np.int32)
        dist = np.empty((nq, k), dtype=np.float32)
        lat = C.c_double()
        results.append(L.lib.da_nn_server_wait_s(srv.h, rid, L.ptr(ind), L.ptr(dist),
                                                 C.byref(lat)))

    th = [threading.Thread(target=waiter) for _ in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert sorted(results) == [L.CODE["success"], L.CODE["invalid_input"]]
    srv._k.pop(rid)
    srv.close()


@pytest.mark.parametrize("max_bytes", [64 << 20, 256 << 20])
def test_device_bytes_stay_within_the_limit(max_bytes):
    """Batches of 1,000,000 rows, hit bits of 134 KB a query: with 256 MB a slot searches them in
    blocks, with 64 MB not even one group of 256 queries fits and the fused tile serves. The
    training operand (64 MB) is laid out when the server is created."""
    rng = np.random.default_rng(36)
    means = rng.uniform(-10, 10, (32, 16))
    Xt = (means[rng.integers(0, 32, 1000000)] +
          rng.standard_normal((1000000, 16))).astype(np.float32)
    Q = (means[rng.integers(0, 32, 9000)] + rng.standard_normal((9000, 16))).astype(np.float32)
    nn = aoclda.neighbors.nearest_neighbors().fit(Xt)

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert L.lib.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    srv = nn_server(nn, max_batch_queries=4096, max_device_bytes=max_bytes)
    before = free()
    cuts = [0, 1, 700, 4796, 9000]
    ks = [10, 1, 100, 16]
    got = []
    for _ in range(2):
        ids = [srv.submit(Q[a:b], k) for a, b, k in zip(cuts, cuts[1:], ks)]
        got = [srv.wait(r) for r in ids]
    # 24 MB: allocations are rounded up to 2 MB, and the selection's own scratch
    assert before - free() < max_bytes + (24 << 20)
    srv.close()
    for (dist, ind, _), a, b, k in zip(got, cuts, cuts[1:], ks):
        de, ie = nn.kneighbors(Q[a:b], n_neighbors=k)
        np.testing.assert_array_equal(ind, ie)
        np.testing.assert_array_equal(dist, de)


@pytest.mark.parametrize("max_bytes", [64 << 20, 256 << 20])
@pytest.mark.parametrize("metric", ["euclidean", "cosine"])
def test_device_bytes_of_wide_rows(metric, max_bytes):
    """150,000 rows of 200 features: approximate scores in blocks of 128 queries (77 MB) with 256 MB,
    key tiles a few queries at a time with 64 MB; clusters so tight that every query is searched
    again."""
    rng = np.random.default_rng(37)
    means = rng.uniform(-10, 10, (32, 200))
    lab, qlab = rng.integers(0, 32, 150000), rng.integers(0, 32, 700)
    for sigma in (1.0, 1e-3):
        Xt = (means[lab] + sigma * rng.standard_normal((150000, 200))).astype(np.float32)
        Q = (means[qlab] + sigma * rng.standard_normal((700, 200))).astype(np.float32)
        nn = aoclda.neighbors.nearest_neighbors(metric=metric, algorithm="brute").fit(Xt)

        def free():
            a, b = C.c_size_t(), C.c_size_t()
            assert L.lib.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
            return a.value

        srv = nn_server(nn, max_batch_queries=1024, max_device_bytes=max_bytes)
        before = free()
        dist, ind, _ = srv.wait(srv.submit(Q, 10))
        assert before - free() < max_bytes + (24 << 20)
        srv.close()
        de, ie = nn.kneighbors(Q, n_neighbors=10)
        np.testing.assert_array_equal(ind, ie)
        np.testing.assert_array_equal(dist, de)


@pytest.mark.parametrize("n,d", [(47000, 8), (31531, 1), (3000, 5)])
def test_few_bytes_and_queries_the_hit_bits_leave(n, d):
    """Key tiles of a few rows at a time or, beyond eight of those, the fused tile: the results of
    the handle's own search."""
    rng = np.random.default_rng(d)
    means = rng.uniform(-10, 10, (16, d))
    X = (means[rng.integers(0, 16, n)] + 0.1 * rng.standard_normal((n, d))).astype(np.float32)
    nn = aoclda.neighbors.nearest_neighbors(metric="euclidean").fit(X)
    qs = [(means[rng.integers(0, 16, q)] + 0.1 * rng.standard_normal((q, d))).astype(np.float32)
          for q in (1, 40, 130, 300, 2200)]
    want = [nn.kneighbors(q, n_neighbors=9) for q in qs]
    srv = nn_server(nn, max_batch_queries=4096, max_device_bytes=64 << 20)
    for _ in range(2):
        for (wd, wi), rid in zip(want, [srv.submit(q, 9) for q in qs]):
            dist, ind, _ = srv.wait(rid)
            np.testing.assert_array_equal(ind, wi)
            np.testing.assert_array_equal(dist, wd)
    srv.close()
