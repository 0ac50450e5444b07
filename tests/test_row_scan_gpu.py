"""The row-per-lane scans (knn_rows.hip): the vector-ALU metrics at every batch size, packed Hamming in
small batches, and the fp4 Hamming round plans.

A score's terms are summed in one order whatever the batch, so a query gets the same ids and the same
distances, bit for bit, whether it is searched alone or within a large batch.  Batches of up to 128
queries take the small-batch round plan and count candidates on spread counters; the batch of 300 they
are compared with takes the growing plan, and is held to the oracle.  Sizes sit at the edges of the
kernels: query tiles of 4 and 16, 128 and 129 queries, 32-dimension chunks and halves of 16, the two
sums' boundary at 64 and 128 dimensions, workgroups of 256 rows, bases of one dense round (16,384 rows
in the small plan, 2,048 in the other) and of several."""
import numpy as np
import pytest

from knn_check import check_knn

pytestmark = pytest.mark.gpu

ORACLE = {"Manhattan": "l1", "Minkowski": "minkowski", "Chebyshev": "linf", "Hamming": "hamming",
          "Mahalanobis": "mahalanobis", "Jaccard": "jaccard", "Hellinger": "hellinger"}


@pytest.fixture(scope="module")
def vh():
    import vector_hip

    assert vector_hip.CudaDeviceContext.device_count() >= 1
    return vector_hip


@pytest.mark.parametrize("metric", list(ORACLE))
@pytest.mark.parametrize("n,dim,k", [(3, 5, 10), (257, 32, 1), (8193, 33, 7), (20_001, 65, 100), (16_385, 128, 10),
                                     (140_000, 129, 10), (9000, 200, 300)])
def test_every_batch_size_agrees(vh, oracle, metric, n, dim, k):
    rng = np.random.default_rng(n + dim)
    base = rng.uniform(-1, 1, (n, dim)).astype(np.float32)
    base[rng.integers(0, n, n // 3)] = base[rng.integers(0, n, n // 3)]  # equal rows: ties by id
    if metric == "Hamming":
        base = np.round(base * 2)
    q = np.concatenate([base[:2], rng.uniform(-1, 1, (298, dim)).astype(np.float32)])
    eng = vh.CudaKnnEngine(base, dim, vh.DistanceMetric[metric])
    ids, dist, lens = eng.search_batch_arrays(q, k)
    kk = min(k, n)
    held = [0, 1, 2, 7, 128, 299]
    # sums of up to 200 terms in another order than the oracle's, and cbrt / sqrt of them
    check_knn(oracle, base, q[held], ids[held], dist[held], k, ORACLE[metric], rtol=2e-5, atol=2e-6)
    for nq in (1, 4, 5, 16, 17, 64, 128, 129):
        i2, d2, l2 = eng.search_batch_arrays(q[:nq], k)
        np.testing.assert_array_equal(i2[:, :kk], ids[:nq, :kk])
        np.testing.assert_array_equal(d2[:, :kk], dist[:nq, :kk])
        np.testing.assert_array_equal(l2, lens[:nq])


# one dense round in the small plan and several in the other; dense and filter rounds in both
@pytest.mark.parametrize("n,share", [(9000, 0.999), (60_000, 0.9998), (60_000, 0.5)])
@pytest.mark.parametrize("metric", ["Manhattan", "Minkowski"])
def test_rows_and_queries_with_nan(vh, metric, n, share):
    """A row with a NaN never appears and a query with one finds nothing, in small and large batches alike,
    whether the rows without are fewer than k or many, in the first round or in later ones."""
    rng = np.random.default_rng(3)
    base = rng.uniform(-1, 1, (n, 40)).astype(np.float32)
    bad = rng.random(n) < share
    base[bad, 7] = np.nan
    q = rng.uniform(-1, 1, (300, 40)).astype(np.float32)
    q[1, 0] = np.nan
    eng = vh.CudaKnnEngine(base, 40, vh.DistanceMetric[metric])
    ids, dist, _ = eng.search_batch_arrays(q, 30)
    good = np.flatnonzero(~bad)
    assert good.size > 0
    found = min(30, good.size)
    p = 1 if metric == "Manhattan" else 3
    for r in (0, 2, 299):
        assert np.all(np.isin(ids[r, :found], good)) and len(set(ids[r, :found].tolist())) == found
        assert np.all(ids[r, found:] == 0xFFFFFFFF) and np.all(np.isnan(dist[r, found:]))
        want = np.sort((np.abs(base[good].astype(np.float64) - q[r]) ** p).sum(1) ** (1 / p))[:found]
        np.testing.assert_allclose(dist[r, :found], want, rtol=1e-5)  # 40 terms in 32 bits
    assert np.all(ids[1] == 0xFFFFFFFF)
    for nq in (2, 16, 33, 128, 129):
        i2, d2, _ = eng.search_batch_arrays(q[:nq], 30)
        np.testing.assert_array_equal(i2, ids[:nq])
        np.testing.assert_array_equal(d2, dist[:nq])


@pytest.mark.parametrize("words", [1, 2, 3, 8, 9, 32])
@pytest.mark.parametrize("n,k", [(5, 10), (257, 3), (20_000, 100), (300_001, 10)])
def test_hamming_small_batches(vh, words, n, k):
    rng = np.random.default_rng(words * 1000 + n)
    codes = rng.integers(0, 1 << 32, (n, words), dtype=np.uint64).astype(np.uint32)
    codes[rng.integers(0, n, n // 3)] = codes[0]  # massive ties
    q = np.concatenate([codes[:2], rng.integers(0, 1 << 32, (68, words), dtype=np.uint64).astype(np.uint32)])
    eng = vh.HammingKnnEngine(codes)
    ids, dist, _ = eng.search_batch_arrays(q, k)
    kk = min(k, n)
    d0 = np.array([np.sum([bin(int(w)).count("1") for w in q[0] ^ codes[i]]) for i in ids[0, :kk]])
    np.testing.assert_array_equal(dist[0, :kk], d0)
    for nq in (1, 4, 5, 17, 64):
        i2, d2, _ = eng.search_batch_arrays(q[:nq], k)
        np.testing.assert_array_equal(i2[:, :kk], ids[:nq, :kk])
        np.testing.assert_array_equal(d2[:, :kk], dist[:nq, :kk])


@pytest.mark.parametrize("words,n,nq,k", [(2, 30_001, 7168, 1), (8, 30_001, 7169, 1), (32, 30_001, 7169, 40),
                                          (8, 40_001, 5120, 1), (8, 40_001, 5121, 1), (2, 40_001, 5121, 70),
                                          (32, 40_001, 2047, 1), (16, 40_001, 2048, 10), (8, 40_001, 14_337, 1)])
def test_hamming_large_batches(vh, monkeypatch, words, n, nq, k):
    """Both sides of the batch sizes from which the fp4 scan's first round has 1,024 or 512 rows, and k whose
    20 k rows are more than that; the popcount batch kernel is the reference."""
    rng = np.random.default_rng(words + nq)
    codes = rng.integers(0, 1 << 32, (n, words), dtype=np.uint64).astype(np.uint32)
    q = rng.integers(0, 1 << 32, (nq, words), dtype=np.uint64).astype(np.uint32)
    ids, dist, _ = vh.HammingKnnEngine(codes).search_batch_arrays(q, k)
    monkeypatch.setenv("VHIP_HAMMING_KERNEL", "popcount")
    i2, d2, _ = vh.HammingKnnEngine(codes).search_batch_arrays(q, k)
    np.testing.assert_array_equal(ids, i2)
    np.testing.assert_array_equal(dist, d2)


@pytest.mark.parametrize("words", [2, 8, 32])
@pytest.mark.parametrize("nq", [17, 128, 129, 256])
def test_hamming_mid_batches(vh, monkeypatch, words, nq):
    """Mid-size batches on the fp4 matrix cores take the small-batch round plan (dense rounds cut into
    512-row items); the popcount batch kernel has the growing plan and is the reference here."""
    rng = np.random.default_rng(words + nq)
    codes = rng.integers(0, 1 << 32, (150_001, words), dtype=np.uint64).astype(np.uint32)
    q = rng.integers(0, 1 << 32, (nq, words), dtype=np.uint64).astype(np.uint32)
    ids, dist, _ = vh.HammingKnnEngine(codes).search_batch_arrays(q, 30)
    monkeypatch.setenv("VHIP_HAMMING_KERNEL", "popcount")
    i2, d2, _ = vh.HammingKnnEngine(codes).search_batch_arrays(q, 30)
    np.testing.assert_array_equal(ids, i2)
    np.testing.assert_array_equal(dist, d2)
