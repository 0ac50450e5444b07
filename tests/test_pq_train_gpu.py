"""PQ training and encoding of narrow sub-vectors (pq_train.hip), all sub-spaces in one launch.

Training under squared L2 is held to the general k-means engine run on each sub-space by itself, which
it replaces there: on whole-number data whose sums stay exact, the codebooks agree to the last bits of
the centroid division.  Encoding is held to the oracle's argmin in every metric."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def vh():
    import vector_hip

    assert vector_hip.CudaDeviceContext.device_count() >= 1
    return vector_hip


# padded widths 4, 8, 16, 32 and their edges, one and several workgroups, odd cluster counts, n < ks
@pytest.mark.parametrize("n,ds,m,ks,iters", [(1, 1, 1, 4, 2), (255, 3, 2, 7, 3), (513, 4, 1, 1, 2), (3000, 5, 3, 256, 4),
                                             (20_001, 8, 4, 255, 3), (5000, 9, 2, 64, 5), (70_000, 16, 2, 256, 3),
                                             (4097, 17, 2, 33, 4), (9000, 32, 3, 256, 3), (100, 32, 2, 256, 0)])
@pytest.mark.parametrize("given", [True, False])
def test_train_equals_the_general_engine(vh, n, ds, m, ks, iters, given):
    rng = np.random.default_rng(n + ds)
    x = rng.integers(-60, 60, (n, m * ds)).astype(np.float32)
    ek = min(ks, n)
    init = None
    if given:
        init = np.zeros((m, ks, ds), np.float32)
        for j in range(m):
            init[j, :ek] = x[rng.permutation(n)[:ek], j * ds:(j + 1) * ds]
    pq = vh.ProductQuantizer.train(x, m * ds, m, ks, iters, -1.0, seed=11, init_codebooks=init)
    got = pq.codebooks.reshape(m, ks, ds)
    for j in range(m):
        sub = np.ascontiguousarray(x[:, j * ds:(j + 1) * ds])
        st = vh.KMeansState(sub)
        c, _, _ = st.fit(ks, iters, -1.0, init=None if init is None else init[j, :ek], init_mode=vh.INIT_SHUFFLE,
                         seed=11 + 1 + j)
        np.testing.assert_allclose(got[j, :ek], c, rtol=1e-6, atol=1e-6)
        assert not got[j, ek:].any()


def test_sub_spaces_stop_by_themselves(vh):
    """With a tolerance each sub-space stops at its own iteration: the first is at a fixed point from the
    start (one iteration), the second is not."""
    rng = np.random.default_rng(5)
    a = np.repeat(np.array([[0, 0], [100, 0], [0, 100], [100, 100]], np.float32), 500, 0)
    b = rng.integers(0, 1000, (2000, 2)).astype(np.float32)
    x = np.concatenate([a, b], 1)
    init = np.zeros((2, 4, 2), np.float32)
    init[0], init[1] = a[::500], b[:4]
    got = vh.ProductQuantizer.train(x, 4, 2, 4, 40, 1e-4, init_codebooks=init).codebooks.reshape(2, 4, 2)
    np.testing.assert_array_equal(got[0], a[::500])
    c, _, r = vh.KMeansState(np.ascontiguousarray(b)).fit(4, 40, 1e-4, init=b[:4])
    assert 1 < r[2] < 40
    np.testing.assert_allclose(got[1], c, rtol=1e-6)


def test_a_nan_centroid_does_not_keep_a_sub_space_running(vh):
    """A NaN centroid's shift is NaN; as in the general engine it takes no part in the largest shift, so the
    sub-space stops after the first iteration, when the others moved by less than the tolerance."""
    rng = np.random.default_rng(6)
    x = rng.integers(0, 100, (2000, 2)).astype(np.float32)
    x[0, 0] = np.nan  # nearest to no centroid: goes to the first
    init = np.concatenate([[[np.nan, 0.0]], x[1:8]]).astype(np.float32)[None]
    got = vh.ProductQuantizer.train(x, 2, 1, 8, 30, 1e4, init_codebooks=init).codebooks.reshape(8, 2)
    c, _, r = vh.KMeansState(x).fit(8, 30, 1e4, init=init[0])
    assert r[2] == 1
    np.testing.assert_allclose(got[1:], c[1:], rtol=1e-6)


def test_threads_train_with_different_cluster_counts(vh):
    """Trainings that need 39, 65 and 98 KB of LDS a workgroup, at the same time."""
    from concurrent.futures import ThreadPoolExecutor

    rng = np.random.default_rng(9)
    x = rng.integers(-60, 60, (4000, 64)).astype(np.float32)
    jobs = [100, 256, 170, 256, 100, 256, 170, 256]

    def run(ks):
        return vh.ProductQuantizer.train(x, 64, 2, ks, 6, -1.0, seed=3).codebooks

    alone = {ks: run(ks) for ks in set(jobs)}
    with ThreadPoolExecutor(max_workers=4) as ex:
        for _ in range(4):
            for ks, got in zip(jobs, ex.map(run, jobs)):
                np.testing.assert_array_equal(got, alone[ks])


# one sub-space at a time and several uploads (limit 1), groups of like and of unlike size, the limit just
# below what all sub-spaces take
@pytest.mark.parametrize("n,ds,m,ks,limit", [(70_000, 16, 8, 256, 1), (70_000, 16, 8, 256, 30 << 20),
                                             (20_000, 5, 7, 100, 3 << 20), (300, 32, 3, 256, 1), (5000, 1, 64, 16, 2 << 20)])
@pytest.mark.parametrize("tol", [-1.0, 1e-3])
def test_groups_of_sub_spaces(vh, monkeypatch, n, ds, m, ks, limit, tol):
    """Where device memory is short the sub-spaces are trained in groups: the same codebooks, bit for bit."""
    rng = np.random.default_rng(n + m)
    x = rng.standard_normal((n, m * ds)).astype(np.float32)
    whole = vh.ProductQuantizer.train(x, m * ds, m, ks, 4, tol, seed=5).codebooks
    monkeypatch.setenv("VHIP_PQ_TRAIN_BYTES", str(limit))
    np.testing.assert_array_equal(vh.ProductQuantizer.train(x, m * ds, m, ks, 4, tol, seed=5).codebooks, whole)
    x[n // 2, m * ds - 1] = np.inf  # in the last group
    with pytest.raises(vh.InvalidConfig):
        vh.ProductQuantizer.train(x, m * ds, m, ks, 4, tol, seed=5)


def test_training_stays_within_its_memory(vh, monkeypatch):
    """32 sub-spaces of one float, padded to four: 690 MB all at once, 17 MB a sub-space and upload."""
    import ctypes
    import threading

    hip = ctypes.CDLL("libamdhip64.so")

    def free():
        f, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(total)) == 0
        return f.value

    rng = np.random.default_rng(1)
    x = rng.standard_normal((1_000_000, 32)).astype(np.float32)
    vh.ProductQuantizer.train(x[:1000], 32, 32, 16, 1, -1.0)
    monkeypatch.setenv("VHIP_PQ_TRAIN_BYTES", str(64 << 20))
    before, least, done = free(), [1 << 62], threading.Event()

    def watch():
        while not done.is_set():
            least[0] = min(least[0], free())

    t = threading.Thread(target=watch)
    t.start()
    try:
        vh.ProductQuantizer.train(x, 32, 32, 16, 2, -1.0)
    finally:
        done.set()
        t.join()
    used = before - least[0]
    print(f"  training took {used >> 20} MB of device memory at most", flush=True)
    assert 16 << 20 <= used < 150 << 20


def test_infinite_values_are_refused(vh):
    x = np.zeros((300, 8), np.float32)
    x[7, 5] = np.inf
    with pytest.raises(vh.InvalidConfig):
        vh.ProductQuantizer.train(x, 8, 2, 4, 2, -1.0)


@pytest.mark.parametrize("metric", ["l2", "dot", "cosine", "l1", "minkowski", "linf", "hamming", "mahalanobis",
                                    "jaccard", "hellinger"])
@pytest.mark.parametrize("n,ds,m,ks", [(1, 1, 3, 2), (257, 6, 2, 255), (513, 16, 1, 256), (1000, 31, 2, 3)])
def test_encode_narrow(vh, oracle, metric, n, ds, m, ks):
    rng = np.random.default_rng(ds * 100 + ks)
    codes = {"l2": 0, "dot": 1, "cosine": 2, "l1": 3, "minkowski": 4, "linf": 5, "hamming": 6, "mahalanobis": 7,
             "jaccard": 8, "hellinger": 9}
    cb = rng.integers(-5, 6, (m, ks, ds)).astype(np.float32)
    x = rng.integers(-5, 6, (n, m * ds)).astype(np.float32)
    pq = vh.ProductQuantizer(m * ds, m, ks, cb)
    got = pq.encode_batch(x, vh.DistanceMetric(codes[metric]))
    for j in range(m):
        sub, c = np.ascontiguousarray(x[:, j * ds:(j + 1) * ds]), cb[j]
        d = np.stack([oracle.distance_rows(metric, sub, np.repeat(c[t:t + 1], n, 0)) for t in range(ks)], 1)
        best = d.max(1) if metric in ("dot", "cosine") else d.min(1)
        mine = d[np.arange(n), got[:, j]]
        np.testing.assert_allclose(mine, best, rtol=2e-6, atol=2e-6)
        if metric in ("l2", "dot", "l1", "linf", "hamming"):  # exact values: the lowest index among equals
            first = (d.argmax(1) if metric == "dot" else d.argmin(1))
            np.testing.assert_array_equal(got[:, j], first)
