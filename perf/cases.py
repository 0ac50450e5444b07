"""The work that programs have this library do, as cases that can be timed and compared.

Five families, all through the package's public entry points:

* ``knn``      exact search of a query batch over a resident float base (CudaKnnEngine), with queries
               and results in device memory, or in host buffers as the C ABI's first entry point takes them;
* ``hamming``  exact search over packed binary codes (HammingKnnEngine);
* ``kmeans``   training: CudaKMeansEngine.fit from host data with its own seeded k-means++ start
               (``init`` "pp"), or Lloyd iterations on resident points from given centroids ("given");
* ``pq``       product quantizer: training on a sample, then encoding it (ProductQuantizer);
* ``ivfpq``    approximate search of a query batch over a loaded IVF-PQ index (IvfPqIndex).

``listed()`` holds one case for each of the sizes at which these are used; ``draw()`` gives others of
the same ranges: bases from a few thousand rows to a million, rows of 16 to 1,024 floats, batches of one
query to ten thousand, k from 1 to 100.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vector-rs_amd"))
import vector_hip as vh  # noqa: E402

METRICS = {
    "l2": vh.DistanceMetric.L2Squared,
    "dot": vh.DistanceMetric.DotProduct,
    "cosine": vh.DistanceMetric.CosineSimilarity,
    "l1": vh.DistanceMetric.Manhattan,
    "minkowski": vh.DistanceMetric.Minkowski,
    "linf": vh.DistanceMetric.Chebyshev,
    "mahalanobis": vh.DistanceMetric.Mahalanobis,
    "jaccard": vh.DistanceMetric.Jaccard,
    "hellinger": vh.DistanceMetric.Hellinger,
}
GEMM = ("l2", "dot", "cosine")


def listed():
    return [
        # one request of a retrieval service over a small collection of text embeddings: latency alone
        {"name": "knn_cosine_10kx768_q1", "family": "knn", "metric": "cosine", "data": "uniform", "n": 10_000, "d": 768,
         "nq": 1, "k": 10, "buffers": "device"},
        # a service's micro-batch over a million integer image descriptors
        {"name": "knn_l2_1Mx128_q32", "family": "knn", "metric": "l2", "data": "int", "n": 1_000_000, "d": 128,
         "nq": 32, "k": 10, "buffers": "device"},
        # the offline job: exact neighbours of ten thousand descriptors (the benchmark's default workload)
        {"name": "knn_l2_1Mx128_q10k", "family": "knn", "metric": "l2", "data": "int", "n": 1_000_000, "d": 128,
         "nq": 10_000, "k": 100, "buffers": "device"},
        # word-vector width, sizes that are no multiple of anything: maximum inner product of a mid batch
        {"name": "knn_dot_200003x300_q1000", "family": "knn", "metric": "dot", "data": "normal", "n": 200_003, "d": 300,
         "nq": 1000, "k": 20, "buffers": "device"},
        # a micro-batch under a metric that is no matrix product
        {"name": "knn_l1_500kx128_q16", "family": "knn", "metric": "l1", "data": "uniform", "n": 500_000, "d": 128,
         "nq": 16, "k": 10, "buffers": "device"},
        # the same kind of metric for a mid batch with ragged sizes
        {"name": "knn_linf_150001x100_q700", "family": "knn", "metric": "linf", "data": "uniform", "n": 150_001,
         "d": 100, "nq": 700, "k": 10, "buffers": "device"},
        # near-duplicate lookup of a few binary fingerprints
        {"name": "hamming_4Mx256_q16", "family": "hamming", "n": 4_000_000, "bits": 256, "nq": 16, "k": 10},
        # the same collection searched by a large batch
        {"name": "hamming_4Mx256_q4096", "family": "hamming", "n": 4_000_000, "bits": 256, "nq": 4096, "k": 10},
        # training a coarse quantizer on a sample of descriptors in host memory, default start
        {"name": "kmeans_fit_100kx128_k256", "family": "kmeans", "metric": "l2", "data": "int", "init": "pp",
         "n": 100_000, "d": 128, "k": 256, "iters": 10},
        # refining a larger codebook on resident points from centroids at hand
        {"name": "kmeans_lloyd_500kx96_k1024", "family": "kmeans", "metric": "l2", "data": "normal", "init": "given",
         "n": 500_000, "d": 96, "k": 1024, "iters": 5},
        # the product quantizer of an index build: eight sub-spaces of 256 centroids, then the codes
        {"name": "pq_train_encode_65536x128_m8", "family": "pq", "n": 65_536, "d": 128, "m": 8, "ks": 256, "iters": 10},
        # approximate search with the index's default eight-byte codes
        {"name": "ivfpq_400kx128_m8_q2000", "family": "ivfpq", "n": 400_000, "d": 128, "nlist": 512, "m": 8,
         "nprobe": 16, "nq": 2000, "k": 10},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["knn", "knn", "knn_other", "hamming", "kmeans", "pq", "ivfpq"])
    if family in ("knn", "knn_other"):
        gemm = family == "knn"
        metric = rng.choice(GEMM) if gemm else rng.choice([m for m in METRICS if m not in GEMM])
        d = rng.choice([_log(rng, 16, 1024), 32 * rng.randint(1, 32), rng.choice([64, 100, 128, 200, 300, 384, 512, 768, 960])])
        n = min(_log(rng, 2_000, 1_000_000), 150_000_000 // d)
        # at most the largest listed case's time: the other metrics run on the vector units
        nq = max(1, min(_log(rng, 1, 10_000), int((6e11 if gemm else 5e10) / (n * d))))
        data = rng.choice(["int", "normal", "uniform"]) if metric in ("l2", "dot") else "uniform"
        return {"family": "knn", "metric": metric, "data": data, "n": n, "d": d, "nq": nq,
                "k": min(_log(rng, 1, 100), n), "buffers": rng.choice(["device", "device", "host"])}
    if family == "hamming":
        return {"family": "hamming", "n": _log(rng, 20_000, 5_000_000), "bits": rng.choice([64, 128, 256, 512]),
                "nq": _log(rng, 1, 5_000), "k": _log(rng, 1, 100)}
    if family == "kmeans":
        init = rng.choice(["pp", "given"])
        n = _log(rng, 5_000, 200_000)
        return {"family": "kmeans", "metric": "l2", "data": "int" if init == "pp" else "normal", "init": init, "n": n,
                "d": _log(rng, 16, 256), "k": _log(rng, 8, 512 if init == "given" else 128), "iters": rng.randint(3, 8)}
    if family == "pq":
        m = rng.choice([4, 8, 12, 16])
        return {"family": "pq", "n": _log(rng, 4_000, 40_000), "d": m * rng.choice([4, 6, 8, 12, 16]), "m": m,
                "ks": rng.choice([64, 256, 256]), "iters": rng.randint(3, 5)}
    m = rng.choice([4, 8, 8, 12, 16, 32])
    return {"family": "ivfpq", "n": _log(rng, 20_000, 300_000), "d": m * rng.choice([4, 6, 8]), "nlist": _log(rng, 32, 512),
            "m": m, "nprobe": _log(rng, 1, 24), "nq": _log(rng, 1, 3_000), "k": _log(rng, 1, 100)}


# ---- inputs ------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed * 1_000_003 + 17)


def _values(g, rows, d, data):
    """float32 [rows, d] on the GPU: integers in [0, 255], N(0, 1), or uniform in [-1, 1]."""
    if data == "int":
        return torch.randint(0, 256, (rows, d), generator=g, device="cuda", dtype=torch.int32).float()
    if data == "normal":
        return torch.randn((rows, d), generator=g, device="cuda")
    return torch.rand((rows, d), generator=g, device="cuda") * 2 - 1


def _mixture(g, rows, d, components, whole, sigma=1.0):
    """Points around `components` centres ~ N(0, 4 I) with noise N(0, sigma^2 I); `whole`: whole numbers in
    [0, 255], as byte descriptors have.  Also the centres."""
    centres = torch.randn((components, d), generator=g, device="cuda") * 2
    label = torch.randint(0, components, (rows,), generator=g, device="cuda")
    x = centres[label] + torch.randn((rows, d), generator=g, device="cuda") * sigma
    if whole:
        x = (x * 20 + 128).round().clamp(0, 255)
    return x, centres


def _knn_inputs(case, seed):
    g = _gen(seed)
    return _values(g, case["n"], case["d"], case["data"]), _values(g, case["nq"], case["d"], case["data"])


def _hamming_inputs(case, seed):
    """Random codes; each query is a stored code with one bit in eight flipped."""
    g = _gen(seed)
    n, w, nq = case["n"], case["bits"] // 32, case["nq"]
    codes = torch.randint(-2**31, 2**31, (n, w), generator=g, device="cuda", dtype=torch.int32)
    pick = torch.randint(0, n, (nq,), generator=g, device="cuda")
    flip = torch.full((nq, w), -1, dtype=torch.int32, device="cuda")
    for _ in range(3):
        flip &= torch.randint(-2**31, 2**31, (nq, w), generator=g, device="cuda", dtype=torch.int32)
    return codes, codes[pick] ^ flip


def _kmeans_inputs(case, seed):
    g = _gen(seed)
    x, _ = _mixture(g, case["n"], case["d"], max(2, case["k"]), case["data"] == "int")
    start = x[torch.randperm(case["n"], generator=g, device="cuda")[:case["k"]]]
    return x, start


def _pq_inputs(case, seed):
    """Residual-like vectors and a sample of them as the sub-spaces' first centroids, [M, Ks, ds]."""
    g = _gen(seed)
    n, d, m, ks = case["n"], case["d"], case["m"], case["ks"]
    x, _ = _mixture(g, n, d, 256, False)
    rows = x[torch.randperm(n, generator=g, device="cuda")[:ks]]
    return x, rows.view(ks, m, d // m).permute(1, 0, 2).contiguous()


def _nearest(x, c):
    """Row of c nearest to each row of x."""
    out = torch.empty(len(x), dtype=torch.int64, device=x.device)
    cn = c.square().sum(1)
    for s in range(0, len(x), 65_536):
        out[s:s + 65_536] = (cn - 2 * (x[s:s + 65_536] @ c.t())).argmin(1)
    return out


def _ivfpq_inputs(case, seed):
    """The parts of a saved index and a query batch, all from one mixture: coarse centroids (the mixture's
    centres), codebooks (a sample of residuals), each vector's list and code, and its row as its id."""
    g = _gen(seed)
    n, d, nlist, m, nq = case["n"], case["d"], case["nlist"], case["m"], case["nq"]
    x, coarse = _mixture(g, n + nq, d, nlist, False)
    x, q = x[:n], x[n:].contiguous()
    lists = _nearest(x, coarse)
    r = (x - coarse[lists]).view(n, m, d // m)
    books = r[torch.randperm(n, generator=g, device="cuda")[:256]].permute(1, 0, 2).contiguous()
    codes = torch.stack([_nearest(r[:, j].contiguous(), books[j]) for j in range(m)], 1).to(torch.uint8)
    order = torch.sort(lists, stable=True).indices
    sizes = torch.bincount(lists, minlength=nlist)
    return coarse, books, sizes, order, codes[order], q


def _np(t):
    return t.cpu().numpy()


def _out(rows, k, dtype):
    return torch.empty((rows, k), dtype=dtype, device="cuda")


def prepare(case, seed):
    f = case["family"]
    s = {"case": dict(case)}
    if f == "knn":
        base, q = _knn_inputs(case, seed)
        s["engine"] = vh.CudaKnnEngine(_np(base), case["d"], METRICS[case["metric"]])
        if case["buffers"] == "host":
            s["q"] = _np(q)
        else:
            s.update(q=q, ids=_out(case["nq"], case["k"], torch.int32), dist=_out(case["nq"], case["k"], torch.float32))
    elif f == "hamming":
        codes, q = _hamming_inputs(case, seed)
        s["engine"] = vh.HammingKnnEngine(_np(codes).view(np.uint32))
        s.update(q=q, ids=_out(case["nq"], case["k"], torch.int32), dist=_out(case["nq"], case["k"], torch.int32))
    elif f == "kmeans":
        x, start = _kmeans_inputs(case, seed)
        if case["init"] == "pp":
            s["x"] = _np(x)
            s["engine"] = vh.CudaKMeansEngine()
        else:
            s["start"] = _np(start)
            s["state"] = vh.KMeansState(_np(x), METRICS[case["metric"]])
    elif f == "pq":
        x, books = _pq_inputs(case, seed)
        s.update(x=_np(x), books=_np(books))
    else:
        coarse, books, sizes, ids, codes, q = _ivfpq_inputs(case, seed)
        m, d = case["m"], case["d"]
        cfg = vh.IvfPqConfig.new(case["nlist"], case["nprobe"], m)
        pq = vh.ProductQuantizer(d, m, 256, _np(books))
        inv = vh.InvertedIndex.from_csr(_np(sizes).astype(np.uint32), _np(ids).astype(np.uint32), _np(codes), m)
        empty = np.zeros((0, d), np.float32)  # a search reads the codes alone
        s["index"] = vh.IvfPqIndex.from_parts(empty, cfg, _np(coarse), pq, inv, d, vh.DistanceMetric.L2Squared)
        s.update(q=q, ids=_out(case["nq"], case["k"], torch.int32), dist=_out(case["nq"], case["k"], torch.float32),
                 len=torch.empty(case["nq"], dtype=torch.int32, device="cuda"))
    torch.cuda.synchronize()  # the library works on streams of its own
    return s


def run(s):
    c = s["case"]
    f = c["family"]
    if f == "knn" and c["buffers"] == "host":
        ids, dist, _ = s["engine"].search_batch_arrays(s["q"], c["k"])
        return [ids.view(np.int32), dist]
    if f in ("knn", "hamming"):
        s["engine"].search_batch_device(s["q"].data_ptr(), c["nq"], c["k"], s["ids"].data_ptr(), s["dist"].data_ptr())
        return [s["ids"], s["dist"]]
    if f == "kmeans":
        if c["init"] == "pp":
            r, assign = s["engine"].fit(s["x"], c["d"], c["k"], c["iters"], -1.0, METRICS[c["metric"]],
                                        return_assign=True)
            return [r.centroids, assign, r.inertia]
        centroids, assign, r = s["state"].fit(c["k"], c["iters"], -1.0, init=s["start"])
        return [centroids, assign, r[3]]
    if f == "pq":
        pq = vh.ProductQuantizer.train(s["x"], c["d"], c["m"], c["ks"], c["iters"], -1.0, init_codebooks=s["books"])
        return [pq.codebooks, pq.encode_batch(s["x"])]
    s["index"].search_batch_device(s["q"].data_ptr(), c["nq"], c["k"], c["nprobe"], s["ids"].data_ptr(),
                                   s["dist"].data_ptr(), s["len"].data_ptr())
    return [s["ids"], s["dist"], s["len"]]


def work(case):
    """Inputs read once and results written once; a multiply-add (or a subtract and an add or max) is 2."""
    c, f = case, case["family"]
    if f == "knn":
        return {"bytes": 4.0 * c["d"] * (c["n"] + c["nq"]) + 8.0 * c["nq"] * c["k"], "flops": 2.0 * c["n"] * c["d"] * c["nq"]}
    if f == "hamming":
        return {"bytes": c["bits"] / 8.0 * (c["n"] + c["nq"]) + 8.0 * c["nq"] * c["k"],
                "flops": 2.0 * c["n"] * c["bits"] * c["nq"]}
    if f == "kmeans":
        points, centres = 4.0 * c["n"] * c["d"], 4.0 * c["k"] * c["d"]
        start = c["k"] if c["init"] == "pp" else 0  # passes of the k-means++ start: one per centre drawn
        return {"bytes": (start + c["iters"]) * points + 2 * centres + 4.0 * c["n"],
                "flops": 2.0 * c["n"] * c["d"] * (c["k"] * c["iters"] + start)}
    if f == "pq":
        return {"bytes": 4.0 * c["n"] * c["d"] * (c["iters"] + 1) + 8.0 * c["ks"] * c["d"] + c["n"] * c["m"],
                "flops": 2.0 * c["n"] * c["d"] * c["ks"] * (c["iters"] + 1)}
    nprobe = min(c["nprobe"], c["nlist"])
    scanned = c["nq"] * c["n"] * nprobe / c["nlist"]  # codes, were all lists alike
    tables = 2.0 * 256 * c["d"] * c["nq"] * nprobe
    return {"bytes": c["n"] * (c["m"] + 4.0) * min(1.0, c["nq"] * nprobe / c["nlist"]) + 4.0 * c["nq"] * c["d"] + 8.0 * c["nq"] * c["k"],
            "flops": 2.0 * c["nq"] * c["nlist"] * c["d"] + tables + c["m"] * scanned}


def tolerance(case):
    f = case["family"]
    if f == "hamming":
        return "exact"
    if f == "knn":
        if case["metric"] == "l2" and case["data"] == "int":
            return {"rel": 1e-6, "differ": 0.0}
        # neighbours whose distances agree to a few units in the last place may change places
        return {"rel": 1e-6, "max": 1e-5, "differ": 1e-3}
    if f == "kmeans":
        # a point between two centres goes with the last bit, and takes its centres along
        return {"rel": 1e-3, "max": 0.1, "differ": 1e-3}
    if f == "pq":  # the same, with few values to a centre
        return {"rel": 3e-3, "max": 0.1, "differ": 1e-3}
    return {"rel": 1e-6, "max": 1e-5, "differ": 1e-3}


# ---- the same results in 64 bits ---------------------------------------------------------------
def _distances(metric, q, x):
    """float64 metric values [nq, n]."""
    if metric in ("l2", "mahalanobis"):
        v = (q.square().sum(1)[:, None] + x.square().sum(1) - 2 * (q @ x.t())).clamp(min=0)
        return v.sqrt() if metric == "mahalanobis" else v
    if metric == "dot":
        return q @ x.t()
    if metric == "cosine":
        return (q @ x.t()) / (q.norm(dim=1)[:, None] * x.norm(dim=1))
    if metric == "l1":
        return _pairwise(q, x, lambda a, b: (a - b).abs().sum(2))
    if metric == "minkowski":
        return _pairwise(q, x, lambda a, b: (a - b).abs().pow(3).sum(2).pow(1 / 3))
    if metric == "linf":
        return _pairwise(q, x, lambda a, b: (a - b).abs().amax(2))
    if metric == "hellinger":
        return _pairwise(q.abs().sqrt(), x.abs().sqrt(), lambda a, b: ((a - b).square().sum(2) / 2).sqrt())
    return _pairwise(q.abs(), x.abs(), lambda a, b: 1 - torch.minimum(a, b).sum(2) / torch.maximum(a, b).sum(2))


def _pairwise(q, x, f):
    """f of every pair, over blocks of x that keep the [nq, block, d] differences within memory."""
    step = max(1, 400_000_000 // (q.shape[0] * q.shape[1]))
    return torch.cat([f(q[:, None], x[None, s:s + step]) for s in range(0, len(x), step)], 1)


def _best(v, k):
    """The k least of each row of v, least first and lower index first where equal: (index, value)."""
    k = min(k, v.shape[1])
    kth = torch.topk(v, k, dim=1, largest=False, sorted=True).values[:, -1:]
    room = min(v.shape[1], k + 64)  # ties with the k-th: the lowest indices among them
    val, idx = torch.topk(v, room, dim=1, largest=False, sorted=True)
    idx = torch.where(val <= kth, idx, v.shape[1])
    idx, o = torch.sort(idx, dim=1, stable=True)
    val, o2 = torch.sort(torch.gather(val, 1, o), dim=1, stable=True)
    return torch.gather(idx, 1, o2)[:, :k], val[:, :k]


def _exact_knn(case, seed):
    base, q = _knn_inputs(case, seed)
    higher = case["metric"] in ("dot", "cosine")
    x, ids, dist = base.double(), [], []
    step = max(1, min(case["nq"], 100_000_000 // case["n"]))
    for s in range(0, case["nq"], step):
        v = _distances(case["metric"], q[s:s + step].double(), x)
        i, d = _best(-v if higher else v, case["k"])
        ids.append(i)
        dist.append(-d if higher else d)
    return [torch.cat(ids).to(torch.int32), torch.cat(dist)]


def _draws(seed, count):
    """The seeded 64-bit draws of the k-means++ start: the published splitmix64 sequence."""
    mask, st, out = (1 << 64) - 1, seed, []
    for _ in range(count):
        st = (st + 0x9E3779B97F4A7C15) & mask
        z = ((st ^ (st >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        out.append(z ^ (z >> 31))
    return out


def _plus_plus(x, k, seed=42):
    """Each next centre is the first point of positive weight at which the running sum of the squared
    distances to the centres so far reaches u times their total (exact: whole numbers)."""
    draws, n = _draws(seed, k), len(x)
    at = draws[0] % n
    picks, least = [at], torch.full((n,), math.inf, dtype=torch.float64, device=x.device)
    for j in range(1, k):
        least = torch.minimum(least, (x - x[at]).square().sum(1))
        run_sum = least.cumsum(0)
        total = float(run_sum[-1])
        if total <= 1e-6:
            at = draws[j] % n
        else:
            reach = (run_sum >= (draws[j] >> 11) * 2.0**-53 * total) & (least > 0)
            at = int(reach.to(torch.int8).argmax())
        picks.append(at)
    return x[picks]


def _lloyd(x, c, iters):
    """(centroids after the last update, the assignment it used, its inertia) in 64 bits."""
    for _ in range(iters):
        a = torch.empty(len(x), dtype=torch.int64, device=x.device)
        least = torch.empty(len(x), dtype=x.dtype, device=x.device)
        xn, cn = x.square().sum(1), c.square().sum(1)
        for s in range(0, len(x), 65_536):
            v = xn[s:s + 65_536, None] + cn - 2 * (x[s:s + 65_536] @ c.t())
            least[s:s + 65_536], a[s:s + 65_536] = v.min(1)
        count = torch.bincount(a, minlength=len(c)).to(x.dtype)
        total = torch.zeros_like(c).index_add_(0, a, x)
        c = torch.where(count[:, None] > 0, total / count.clamp(min=1)[:, None], c)
    return c, a, least.clamp(min=0).sum()


def _exact_kmeans(case, seed):
    x, start = _kmeans_inputs(case, seed)
    x = x.double()
    c = _plus_plus(x, case["k"]) if case["init"] == "pp" else start.double()
    c, a, inertia = _lloyd(x, c, case["iters"])
    return [c, a.to(torch.int32), float(inertia)]


def _exact_pq(case, seed):
    x, books = _pq_inputs(case, seed)
    m, ks, ds = books.shape
    out, codes = [], []
    for j in range(m):
        xs = x[:, j * ds:(j + 1) * ds].double()
        c = _lloyd(xs, books[j].double(), case["iters"])[0]
        out.append(c.reshape(-1))
        codes.append(_nearest(xs, c))
    return [torch.cat(out), torch.stack(codes, 1).to(torch.uint8)]


def _exact_ivfpq(case, seed):
    coarse, books, sizes, ids, codes, q = _ivfpq_inputs(case, seed)
    nlist, m, k, nq = case["nlist"], case["m"], case["k"], case["nq"]
    probes = _best(_distances("l2", q.double(), coarse.double()), case["nprobe"])[0]
    ends = sizes.cumsum(0).tolist()
    width = max(1, min(k, int(sizes.max())))
    best_d = torch.full((nq, probes.shape[1], width), math.inf, dtype=torch.float64, device="cuda")
    best_i = torch.full((nq, probes.shape[1], width), 2**31 - 1, dtype=torch.int64, device="cuda")
    for c in range(nlist):
        lo, hi = (ends[c - 1] if c else 0), ends[c]
        who = (probes == c).nonzero()
        if lo == hi or not len(who):
            continue
        r = (q[who[:, 0]].double() - coarse[c].double()).view(-1, m, 1, books.shape[2])
        table = (r - books.double()).square().sum(3)  # [queries, M, 256]
        v = torch.zeros((len(who), hi - lo), dtype=torch.float64, device="cuda")
        for j in range(m):
            v += table[:, j][:, codes[lo:hi, j].long()]
        i, d = _best(v, width)  # a list holds its ids ascending
        best_d[who[:, 0], who[:, 1], :d.shape[1]] = d
        best_i[who[:, 0], who[:, 1], :d.shape[1]] = ids[lo:hi][i]
    d, i = best_d.view(nq, -1), best_i.view(nq, -1)
    i, o = torch.sort(i, dim=1, stable=True)
    d, o2 = torch.sort(torch.gather(d, 1, o), dim=1, stable=True)
    i = torch.gather(i, 1, o2)
    if d.shape[1] < k:
        d = torch.nn.functional.pad(d, (0, k - d.shape[1]), value=math.inf)
        i = torch.nn.functional.pad(i, (0, k - i.shape[1]), value=-1)
    d, i = d[:, :k], i[:, :k]
    found = torch.isfinite(d)
    count = sizes[probes].sum(1).clamp(max=k)
    return [torch.where(found, i, -1).to(torch.int32), torch.where(found, d, math.nan), count.to(torch.int32)]


def exact(case, seed):
    f = case["family"]
    if f == "knn":
        return _exact_knn(case, seed)
    if f == "hamming":
        return None  # whole numbers
    if f == "kmeans":
        return _exact_kmeans(case, seed)
    return _exact_pq(case, seed) if f == "pq" else _exact_ivfpq(case, seed)
