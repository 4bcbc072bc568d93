"""Performance cases of the distance path: k-nearest neighbours, pairwise distances, k-means,
batched k-means, DBSCAN and IVF-Flat search, each through the entry points that a user's program
calls (the Python front end on host arrays, the C API on device pointers), from the smallest
calls, where launches and latency count, to the largest resident workloads.

listed() holds the fixed cases, draw(rng) makes further ones of the same ranges, prepare() builds
what a program has in hand before the call, run() makes one pass, exact() states the result in
64-bit torch without this package, work() the bytes and operations a pass cannot do without and
tolerance() what the data types allow.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "aocl-data-analytics_amd"))

import aoclda  # noqa: E402
from aoclda import _lib as L  # noqa: E402

DEVICE = "cuda"
TORCH_TYPE = {"float32": torch.float32, "float64": torch.float64}


# ---- cases ----------------------------------------------------------------------------------

def listed():
    return [
        # A small table of numeric records, looked up with the defaults (double precision, host
        # arrays): latency of the whole call.
        dict(name="knn_table_fp64", kind="knn", n=2125, d=20, nq=2068, k=5, dtype="float64",
             precision="working", metric="euclidean", host=True, data="mixture"),
        # The headline search: device-resident queries, centred fp16 operands, exact results.
        dict(name="knn_fp16c", kind="knn", n=200000, d=128, nq=20000, k=10, dtype="float32",
             precision="fp16c", metric="euclidean", host=False, data="mixture"),
        # The default operand precision (fp32) with ragged sizes and host arrays.
        dict(name="knn_fp32", kind="knn", n=100003, d=100, nq=10007, k=20, dtype="float32",
             precision="working", metric="euclidean", host=True, data="mixture"),
        # One batch of a search service over a large index of unit rows, long lists.
        dict(name="knn_service", kind="knn", n=2000000, d=96, nq=1024, k=100, dtype="float32",
             precision="fp16", metric="euclidean", host=False, data="unit"),
        # Wide rows (flattened images, embeddings).
        dict(name="knn_wide", kind="knn", n=60000, d=784, nq=2000, k=5, dtype="float32",
             precision="working", metric="euclidean", host=True, data="mixture"),
        # A small distance matrix in double precision on host arrays.
        dict(name="pairwise_fp64", kind="pairwise", m=2000, n=1500, d=64, dtype="float64",
             metric="euclidean", host=True),
        # A large distance matrix of device-resident rows.
        dict(name="pairwise_fp32", kind="pairwise", m=8192, n=8192, d=256, dtype="float32",
             metric="euclidean", host=False),
        # A large clustering, the data resident in the handle (one k-means++ start).
        dict(name="kmeans_large", kind="kmeans", n=2000000, d=32, k=256, dtype="float32",
             precision="working", init="k-means++", n_init=1, max_iter=25, tol=0.0, host=False),
        # An ordinary clustering with the defaults (ten k-means++ starts, double precision),
        # then the labels of new rows.
        dict(name="kmeans_small", kind="kmeans", n=20000, d=16, k=8, dtype="float64",
             precision="working", init="k-means++", n_init=10, max_iter=300, tol=1e-4,
             host=True),
        # Many uneven clusterings at once.
        dict(name="kmeans_batch", kind="kmeans_batch", instances=256, n_lo=1000, n_hi=50000,
             k_hi=64, max_iter=15),
        # Density clustering of a point cloud with noise.
        dict(name="dbscan", kind="dbscan", n=100000, d=16, dtype="float32", min_samples=10),
        # Approximate search over inverted lists, host arrays.
        dict(name="ivf", kind="ivf", n=1000000, d=96, n_list=1024, n_probe=16, nq=10000, k=10,
             dtype="float32"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["knn", "knn", "knn_wide", "pairwise", "kmeans", "kmeans", "kmeans_batch",
                       "dbscan", "ivf"])
    if kind == "knn":
        dtype = rng.choice(["float32", "float32", "float64"])
        n = _log(rng, 2000, 200000)
        precision = "working"
        if dtype == "float32":
            precision = rng.choice(["working", "fp16x3", "bf16x3", "fp16c"])
        return dict(kind="knn", n=n, d=rng.randint(3, 128), nq=_log(rng, 16, 10000),
                    k=_log(rng, 1, 100), dtype=dtype, precision=precision, metric="euclidean",
                    host=rng.random() < 0.5, data="mixture")
    if kind == "knn_wide":
        return dict(kind="knn", n=_log(rng, 5000, 60000), d=rng.randint(129, 784),
                    nq=_log(rng, 100, 2000), k=_log(rng, 1, 50), dtype="float32",
                    precision="working",
                    metric=rng.choice(["euclidean", "sqeuclidean", "cosine"]),
                    host=rng.random() < 0.5, data="mixture")
    if kind == "pairwise":
        host = rng.random() < 0.4
        top = 3000 if host else 8192
        return dict(kind="pairwise", m=_log(rng, 200, top), n=_log(rng, 200, top),
                    d=_log(rng, 3, 256),
                    dtype=rng.choice(["float32", "float64"]) if host else "float32",
                    metric=rng.choice(["euclidean", "sqeuclidean", "cosine", "manhattan"]),
                    host=host)
    if kind == "kmeans":
        k = _log(rng, 2, 256)
        return dict(kind="kmeans", n=_log(rng, 5000, 1000000), d=rng.randint(2, 64), k=k,
                    dtype=rng.choice(["float32", "float64"]), precision="working",
                    init=rng.choice(["k-means++", "supplied"]), n_init=1,
                    max_iter=rng.randint(5, 25), tol=rng.choice([0.0, 1e-4]),
                    host=rng.random() < 0.5)
    if kind == "kmeans_batch":
        return dict(kind="kmeans_batch", instances=_log(rng, 16, 256), n_lo=1000,
                    n_hi=_log(rng, 5000, 50000), k_hi=rng.randint(8, 64),
                    max_iter=rng.randint(5, 15))
    if kind == "dbscan":
        return dict(kind="dbscan", n=_log(rng, 5000, 100000), d=rng.randint(3, 32),
                    dtype=rng.choice(["float32", "float64"]), min_samples=rng.randint(4, 20))
    n_list = _log(rng, 128, 1024)
    return dict(kind="ivf", n=_log(rng, 200000, 1000000), d=rng.randint(16, 128), n_list=n_list,
                n_probe=rng.randint(4, 16), nq=_log(rng, 500, 10000), k=_log(rng, 1, 20),
                dtype="float32")


# ---- inputs ---------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) * 1000003 + 17)
    return g


def _uniform(g, shape, lo, hi, dtype=torch.float32):
    return torch.rand(shape, generator=g, device=DEVICE, dtype=dtype) * (hi - lo) + lo


def _normal(g, shape, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=dtype)


def _pick(g, count, n):
    return torch.randint(0, count, (n,), generator=g, device=DEVICE)


def _mixture(g, means, n, sigma):
    """n rows about randomly chosen means."""
    return means[_pick(g, means.shape[0], n)] + sigma * _normal(g, (n, means.shape[1]),
                                                                means.dtype)


def _knn_inputs(case, seed):
    """Training rows and queries: a 64-component Gaussian mixture (means U[-10, 10], sigma 1), or
    unit-normalised rows of a 1,024-component one (means N(0, 1), sigma 0.25)."""
    g, t = _gen(seed), TORCH_TYPE[case["dtype"]]
    if case["data"] == "unit":
        means = _normal(g, (1024, case["d"]), t)
        X = _mixture(g, means, case["n"], 0.25)
        Q = _mixture(g, means, case["nq"], 0.25)
        X /= X.norm(dim=1, keepdim=True)
        Q /= Q.norm(dim=1, keepdim=True)
        return X, Q
    means = _uniform(g, (64, case["d"]), -10, 10, t)
    return _mixture(g, means, case["n"], 1.0), _mixture(g, means, case["nq"], 1.0)


def _pairwise_inputs(case, seed):
    g, t = _gen(seed), TORCH_TYPE[case["dtype"]]
    return (_uniform(g, (case["m"], case["d"]), 0, 1, t),
            _uniform(g, (case["n"], case["d"]), 0, 1, t))


def _kmeans_inputs(case, seed):
    """Blobs of unequal spread, one per cluster (means U[-20, 20], sigma U[0.5, 2]); the supplied
    centres are rows of the data, the new rows come from the same blobs."""
    g, t = _gen(seed), TORCH_TYPE[case["dtype"]]
    k, d = case["k"], case["d"]
    means = _uniform(g, (k, d), -20, 20, t)
    sigma = _uniform(g, (k, 1), 0.5, 2.0, t)

    def rows(n):
        lab = _pick(g, k, n)
        return means[lab] + sigma[lab] * _normal(g, (n, d), t)

    X = rows(case["n"])
    new = rows(max(1, case["n"] // 4))
    return X, X[:k].clone(), new


def _batch_shapes(case):
    """Rows, features and clusters of each instance: a property of the case, not of the seed."""
    r = np.random.default_rng([case["instances"], case["n_hi"], case["k_hi"]])
    ni = case["instances"]
    n = np.floor(np.exp(r.uniform(math.log(case["n_lo"]), math.log(case["n_hi"]), ni)))
    d = r.choice([8, 16, 32, 64], ni)
    k = r.integers(4, case["k_hi"] + 1, ni)
    return n.astype(np.int32), d.astype(np.int32), k.astype(np.int32)


def _batch_inputs(case, seed):
    n, d, k = _batch_shapes(case)
    g = _gen(seed)
    xs, cs = [], []
    for ni, di, ki in zip(n.tolist(), d.tolist(), k.tolist()):
        X = _mixture(g, _uniform(g, (ki, di), -10, 10), ni, 1.0)
        xs.append(X)
        cs.append(X[:ki])
    return n, d, k, xs, cs


def _dbscan_inputs(case, seed):
    """32 blobs (means U[-10, 10], sigma 0.5) and 5% noise in [-12, 12]; eps grows with the
    distance between two points of a blob."""
    g, t = _gen(seed), TORCH_TYPE[case["dtype"]]
    n, d = case["n"], case["d"]
    nb = n - n // 20
    X = torch.cat([_mixture(g, _uniform(g, (32, d), -10, 10, t), nb, 0.5),
                   _uniform(g, (n - nb, d), -12, 12, t)])
    return X[torch.randperm(n, generator=g, device=DEVICE)], 0.45 * math.sqrt(d)


def _ivf_inputs(case, seed):
    """A 1,024-component Gaussian mixture (means U[-4, 4], sigma 1)."""
    g, t = _gen(seed), TORCH_TYPE[case["dtype"]]
    means = _uniform(g, (1024, case["d"]), -4, 4, t)
    return _mixture(g, means, case["n"], 1.0), _mixture(g, means, case["nq"], 1.0)


def _host(x):
    return np.ascontiguousarray(x.cpu().numpy())


def _ptr(t):
    return C.c_void_p(t.data_ptr())


# ---- what a program has in hand, and one pass -------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "knn":
        X, Q = _knn_inputs(case, seed)
        s["nn"] = aoclda.neighbors.nearest_neighbors(
            n_neighbors=case["k"], metric=case["metric"], precision=case["precision"],
            algorithm="brute").fit(_host(X))
        if case["host"]:
            s["Q"] = _host(Q)
        else:
            s["Q"] = Q
            s["ind"] = torch.zeros((case["nq"], case["k"]), dtype=torch.int32, device=DEVICE)
            s["dist"] = torch.zeros((case["nq"], case["k"]), dtype=Q.dtype, device=DEVICE)
    elif kind == "pairwise":
        X, Y = _pairwise_inputs(case, seed)
        if case["host"]:
            s["X"], s["Y"] = _host(X), _host(Y)
        else:
            s["X"], s["Y"] = X, Y
            s["D"] = torch.zeros((case["m"], case["n"]), dtype=X.dtype, device=DEVICE)
    elif kind == "kmeans":
        X, C0, new = _kmeans_inputs(case, seed)
        s["km"] = aoclda.clustering.kmeans(
            n_clusters=case["k"], initialization_method=case["init"],
            C=_host(C0) if case["init"] == "supplied" else None, n_init=case["n_init"],
            max_iter=case["max_iter"], seed=42, tol=case["tol"], precision=case["precision"])
        s["X"], s["new"] = _host(X), _host(new)
        if not case["host"]:
            # The data go to the handle once; later passes compute on it.
            short = aoclda.clustering.kmeans(n_clusters=case["k"], initialization_method="random",
                                             n_init=1, max_iter=1, seed=42, tol=0.0,
                                             precision=case["precision"])
            short.fit(s["X"])
            h = short._h
            h.set_string("initialization method", case["init"])
            h.set_int("n_init", case["n_init"])
            h.set_int("max_iter", case["max_iter"])
            h.set_real("convergence tolerance", case["tol"])
            if case["init"] == "supplied":
                s["C0"] = _host(C0)
                h.call("da_kmeans_set_init_centres", L.ptr(s["C0"]), case["d"])
            s["km"] = short
    elif kind == "kmeans_batch":
        n, d, k, xs, cs = _batch_inputs(case, seed)
        s["n"], s["d"], s["k"] = n, d, k
        s["X"] = torch.cat([x.reshape(-1) for x in xs])
        s["C0"] = torch.cat([c.reshape(-1) for c in cs])
        s["C"] = s["C0"].clone()
        s["labels"] = torch.zeros(int(n.sum()), dtype=torch.int32, device=DEVICE)
    elif kind == "dbscan":
        X, eps = _dbscan_inputs(case, seed)
        s["X"], s["eps"] = _host(X), eps
    elif kind == "ivf":
        X, Q = _ivf_inputs(case, seed)
        s["ann"] = aoclda.neighbors.approximate_neighbors(
            n_neighbors=case["k"], n_list=case["n_list"], n_probe=case["n_probe"], kmeans_iter=10,
            seed=0).train_and_add(_host(X))
        s["Q"] = _host(Q)
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "knn":
        nn = s["nn"]
        if case["host"]:
            dist, ind = nn.kneighbors(s["Q"])
            return {"dist": dist, "ind": ind}
        nn.handle.call("da_nn_kneighbors_device", case["nq"], case["d"], _ptr(s["Q"]), case["d"],
                       _ptr(s["ind"]), _ptr(s["dist"]), case["k"], 1)
        return {"dist": s["dist"], "ind": s["ind"]}
    if kind == "pairwise":
        if case["host"]:
            return aoclda.metrics.pairwise_distances(s["X"], s["Y"], metric=case["metric"])
        m, n, d = case["m"], case["n"], case["d"]
        L.check(_noalloc()(L.ROW_MAJOR, m, n, d, _ptr(s["X"]), d, _ptr(s["Y"]), d, _ptr(s["D"]), n,
                           2.0, L.METRICS[case["metric"]]))
        return s["D"]
    if kind == "kmeans":
        km = s["km"]
        if case["host"]:
            km.fit(s["X"])
            return {"centres": km.cluster_centres, "labels": km.labels, "inertia": km.inertia,
                    "new_labels": km.predict(s["new"])}
        km._h.call("da_kmeans_compute", allow=(L.CODE["maxit"],))
        return {"centres": km.cluster_centres, "labels": km.labels, "inertia": km.inertia}
    if kind == "kmeans_batch":
        s["C"].copy_(s["C0"])
        torch.cuda.current_stream().synchronize()  # the call runs on a stream of its own
        ni = case["instances"]
        n_iter = np.zeros(ni, dtype=np.int32)
        inertia = np.zeros(ni, dtype=np.float32)
        L.check(L.lib.da_kmeans_batch_device_s(
            ni, L.ptr(s["n"]), L.ptr(s["d"]), L.ptr(s["k"]), _ptr(s["X"]), _ptr(s["C"]),
            _ptr(s["labels"]), case["max_iter"], 0.0, 0, L.ptr(n_iter), L.ptr(inertia)))
        return {"centres": s["C"], "labels": s["labels"], "inertia": inertia}
    if kind == "dbscan":
        db = aoclda.clustering.DBSCAN(eps=s["eps"], min_samples=case["min_samples"],
                                      algorithm="brute").fit(s["X"])
        core = np.zeros(case["n"], dtype=np.int32)
        core[db.core_sample_indices] = 1
        return {"labels": db.labels, "core": core, "n_clusters": db.n_clusters}
    dist, ind = s["ann"].kneighbors(s["Q"])
    return {"dist": dist, "ind": ind}


def _noalloc():
    """da_pairwise_distances_device_noalloc_s (declared in include/aoclda_amd.h)."""
    f = L.lib.da_pairwise_distances_device_noalloc_s
    i, p = C.c_int32, C.c_void_p
    f.restype = C.c_int
    f.argtypes = [C.c_int, i, i, i, p, i, p, i, p, i, C.c_float, C.c_int]
    return f


# ---- what a pass cannot do without ------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "knn":
        e = 8 if case["dtype"] == "float64" else 4
        n, d, nq, k = case["n"], case["d"], case["nq"], case["k"]
        return {"bytes": e * (n + nq) * d + nq * k * (e + 4), "flops": 2.0 * nq * n * d}
    if kind == "pairwise":
        e = 8 if case["dtype"] == "float64" else 4
        m, n, d = case["m"], case["n"], case["d"]
        return {"bytes": e * ((m + n) * d + m * n), "flops": 2.0 * m * n * d}
    if kind == "kmeans":
        # A pass: each start's k-means++ distances (one centre at a time) and one assignment and
        # update per iteration; the iterations of a run with a tolerance depend on the data and
        # are counted as ten.
        e = 8 if case["dtype"] == "float64" else 4
        n, d, k = case["n"], case["d"], case["k"]
        its = case["max_iter"] if case["tol"] == 0 else min(10, case["max_iter"])
        trials = 2 + int(math.log(k)) if case["init"] == "k-means++" else 0
        per_start = its * (2.0 * n * k * d + n * d) + 2.0 * n * d * trials * (k - 1)
        return {"bytes": e * n * d + 4 * n, "flops": case["n_init"] * per_start}
    if kind == "kmeans_batch":
        n, d, k = (a.astype(np.float64) for a in _batch_shapes(case))
        return {"bytes": float((4 * n * d + 8 * k * d + 4 * n).sum()),
                "flops": float((case["max_iter"] * (2 * n * d * k + n * d)).sum())}
    if kind == "dbscan":
        e = 8 if case["dtype"] == "float64" else 4
        n, d = case["n"], case["d"]
        return {"bytes": e * n * d + 4 * n, "flops": 1.0 * n * n * d}
    n, d, nq = case["n"], case["d"], case["nq"]
    rows = case["n_list"] + case["n_probe"] * n / case["n_list"]
    return {"bytes": 4 * (n + nq) * d + nq * case["k"] * 8, "flops": 2.0 * nq * rows * d}


def tolerance(case):
    kind = case["kind"]
    if kind == "dbscan":
        return "exact"
    # Results are sums in double, rounded once to the working type; whole values (indices, labels)
    # can differ at ties only.
    if kind in ("knn", "ivf"):
        rel = 2e-7 if case["dtype"] == "float32" else 2e-15
        return {"rel": rel, "differ": 2e-5}
    if kind == "pairwise":
        return {"rel": 2e-7 if case["dtype"] == "float32" else 2e-15}
    if kind == "kmeans":
        return {"rel": 4e-7 if case["dtype"] == "float32" else 1e-13, "differ": 2e-5}
    return {"rel": 4e-7, "differ": 2e-5}


# ---- the results in 64 bits --------------------------------------------------------------------

def exact(case, seed):
    kind = case["kind"]
    if kind == "knn":
        return _exact_knn(case, *_knn_inputs(case, seed))
    if kind == "pairwise":
        X, Y = (a.double() for a in _pairwise_inputs(case, seed))
        D = torch.cat([_exact_block(case["metric"], X[i:i + 64], Y)
                       for i in range(0, X.shape[0], 64)])
        return D.cpu().numpy()
    if kind == "kmeans":
        if case["init"] != "supplied" or case["tol"] != 0.0:
            return None  # the starting rows come from the library's own random draws
        X, C0, new = (a.double() for a in _kmeans_inputs(case, seed))
        Cn, lab, inertia = _exact_lloyd(X, C0, case["max_iter"])
        out = {"centres": Cn.cpu().numpy(), "labels": None, "inertia": inertia}
        if case["host"]:
            out["new_labels"] = None
        return out
    if kind == "kmeans_batch":
        _, _, _, xs, cs = _batch_inputs(case, seed)
        cen, inertia = [], []
        for X, C0 in zip(xs, cs):
            Cn, _, v = _exact_lloyd(X.double(), C0.double(), case["max_iter"])
            cen.append(Cn.reshape(-1))
            inertia.append(v)
        return {"centres": torch.cat(cen), "labels": None, "inertia": np.array(inertia)}
    if kind == "ivf":
        # The probed lists hold the nearest rows on this mixture, so the exact neighbours stand
        # for them.
        return _exact_knn(dict(case, metric="sqeuclidean"), *_ivf_inputs(case, seed))
    return None  # DBSCAN's outputs are whole numbers


def _exact_block(metric, X, Y):
    if metric == "manhattan":
        return torch.cdist(X, Y, p=1)
    if metric == "cosine":
        Xn = X / X.norm(dim=1, keepdim=True)
        Yn = Y / Y.norm(dim=1, keepdim=True)
        return 1.0 - Xn @ Yn.T.contiguous()
    D = torch.empty((X.shape[0], Y.shape[0]), dtype=X.dtype, device=X.device)
    step = max(1, (1 << 25) // (X.shape[0] * X.shape[1]))
    for j in range(0, Y.shape[0], step):
        D[:, j:j + step] = (X[:, None, :] - Y[None, j:j + step, :]).square_().sum(2)
    return D.sqrt_() if metric == "euclidean" else D


def _exact_knn(case, X, Q):
    """Distances by matrix products pick a few more neighbours than asked for; direct differences
    of those order them."""
    X, Q = X.double(), Q.double()
    k, metric = case["k"], case["metric"]
    kk = min(X.shape[0], k + 8)
    xs = X.square().sum(1)
    if metric == "cosine":
        X = X / X.norm(dim=1, keepdim=True)
        Q = Q / Q.norm(dim=1, keepdim=True)
    Xt = X.T.contiguous()
    dist, ind = [], []
    step = max(1, (1 << 27) // X.shape[0])
    for i in range(0, Q.shape[0], step):
        q = Q[i:i + step]
        key = q @ Xt
        if metric == "cosine":
            key = 1.0 - key
        else:
            key = xs[None, :] - 2.0 * key
        v, j = torch.topk(key, kk, dim=1, largest=False)
        if metric != "cosine":
            v = torch.stack([(q - X[j[:, t]]).square().sum(1) for t in range(kk)], 1)
        order = torch.argsort(v, dim=1, stable=True)[:, :k]
        dist.append(torch.gather(v, 1, order))
        ind.append(torch.gather(j, 1, order))
    D = torch.cat(dist)
    if metric == "euclidean":
        D = D.sqrt_()
    return {"dist": D.cpu().numpy(), "ind": torch.cat(ind).int().cpu().numpy()}


def _nearest(X, Cn):
    lab = torch.empty(X.shape[0], dtype=torch.int64, device=X.device)
    ct, c2 = Cn.T.contiguous(), Cn.square().sum(1)
    step = 1 << 18
    for i in range(0, X.shape[0], step):
        lab[i:i + step] = torch.argmin(c2[None, :] - 2.0 * (X[i:i + step] @ ct), dim=1)
    return lab


def _exact_lloyd(X, Cn, max_iter):
    k = Cn.shape[0]
    for _ in range(max_iter):
        lab = _nearest(X, Cn)
        cnt = torch.bincount(lab, minlength=k).clamp_(min=1).double()
        S = torch.zeros_like(Cn).index_add_(0, lab, X)
        Cn = S / cnt[:, None]
    lab = _nearest(X, Cn)
    inertia = float((X - Cn[lab]).square().sum())
    return Cn, lab, inertia
