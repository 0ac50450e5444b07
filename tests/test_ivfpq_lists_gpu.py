"""GPU tests of the list-major IVF-PQ scan (16- and 8-byte code rows, 256 sub-centroids, k <= 48).

The list-major search groups the (query, probe) pairs by list and scores each list's codes once
per batch of the queries probing it; the query-major kernel (forced with VHIP_IVFPQ_SCAN=query)
scores them once per probing query.  Both keep the k best (score, id) keys with the same tables
and the same summation order, so their ids and distances must be equal bit for bit.  Shapes
cover skewed and empty lists, lists longer than many ring chunks, more work items than
workgroups, partial items, k from 1 to 48 (the list path's limit; larger k runs query-major,
checked here too), nprobe from 1 to all lists, and the dot-product and cosine table builds.  One
case is also checked against the oracle directly.
"""
import os

import numpy as np
import pytest

from test_ivfpq_gpu import _check_search, _index, _m

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def vh():
    import vector_hip

    assert vector_hip.CudaDeviceContext.device_count() >= 1, "no gfx950 GPU visible"
    return vector_hip


def _skewed_parts(rng, dim, nlist, n, empty=(), integer=False, m_sub=16):
    """Lists of very different sizes (a few hold most rows), some empty."""
    ks, ds = 256, dim // m_sub
    if integer:
        coarse = rng.integers(-4, 5, (nlist, dim)).astype(np.float32)
        cb = rng.integers(-2, 3, m_sub * ks * ds).astype(np.float32)
    else:
        coarse = rng.standard_normal((nlist, dim)).astype(np.float32)
        cb = (0.5 * rng.standard_normal(m_sub * ks * ds)).astype(np.float32)
    weights = rng.exponential(1.0, nlist) ** 3
    weights[list(empty)] = 0.0
    assign = rng.choice(nlist, n, p=weights / weights.sum())
    order = np.argsort(assign, kind="stable")
    sizes = np.bincount(assign, minlength=nlist).astype(np.uint32)
    codes = rng.integers(0, ks, (n, m_sub)).astype(np.uint8)
    return coarse, cb, sizes, order.astype(np.uint32), codes[order]


def _both_paths(ix, qs, k, nprobe):
    old = os.environ.get("VHIP_IVFPQ_SCAN")
    try:
        os.environ.pop("VHIP_IVFPQ_SCAN", None)
        a = ix.search_batch_arrays(qs, k, nprobe)
        os.environ["VHIP_IVFPQ_SCAN"] = "query"
        b = ix.search_batch_arrays(qs, k, nprobe)
    finally:
        if old is None:
            os.environ.pop("VHIP_IVFPQ_SCAN", None)
        else:
            os.environ["VHIP_IVFPQ_SCAN"] = old
    return a, b


def _assert_same(a, b):
    assert np.array_equal(a[2], b[2]), "result counts differ"
    assert np.array_equal(a[0], b[0]), "ids differ"
    assert np.array_equal(a[1].view(np.uint32), b[1].view(np.uint32)), "distances differ"


@pytest.mark.parametrize("dim", [128, 64])
@pytest.mark.parametrize("k,nprobe", [(10, 8), (1, 1), (48, 16), (40, 64), (37, 3), (64, 16), (100, 16)])
def test_lists_match_query_major_l2(vh, dim, k, nprobe):
    rng = np.random.default_rng(dim + 31 * k + nprobe)
    nlist = 64
    parts = _skewed_parts(rng, dim, nlist, 60_000, empty=(5, 17, 40))
    ix = _index(vh, parts, dim, 16, 256, vh.DistanceMetric.L2Squared)
    qs = rng.standard_normal((1500, dim)).astype(np.float32)
    a, b = _both_paths(ix, qs, k, nprobe)
    _assert_same(a, b)
    assert np.all(a[2] <= k)


@pytest.mark.parametrize("metric", ["dot", "cosine"])
def test_lists_match_query_major_inner_product(vh, metric):
    rng = np.random.default_rng(77 if metric == "dot" else 78)
    parts = _skewed_parts(rng, 64, 32, 30_000, empty=(2,))
    ix = _index(vh, parts, 64, 16, 256, _m(vh, metric))
    qs = rng.standard_normal((700, 64)).astype(np.float32)
    for k, nprobe in ((10, 4), (48, 32)):
        a, b = _both_paths(ix, qs, k, nprobe)
        _assert_same(a, b)


def test_lists_integer_exact_against_oracle(vh, oracle):
    """The list-major path on its own against the oracle: integer parts, exact distances."""
    rng = np.random.default_rng(91)
    parts = _skewed_parts(rng, 128, 24, 20_000, empty=(0, 9), integer=True)
    ix = _index(vh, parts, 128, 16, 256, vh.DistanceMetric.L2Squared)
    qs = rng.integers(-4, 5, (40, 128)).astype(np.float32)
    for k, nprobe in ((10, 6), (48, 24), (1, 2), (64, 24), (128, 24)):
        _check_search(vh, oracle, ix, parts, qs, k, nprobe, "l2", 16, 256, exact=True)


def test_lists_repeatable_and_batch_independent(vh):
    rng = np.random.default_rng(92)
    parts = _skewed_parts(rng, 128, 48, 40_000)
    ix = _index(vh, parts, 128, 16, 256, vh.DistanceMetric.L2Squared)
    qs = rng.standard_normal((3000, 128)).astype(np.float32)
    r1 = ix.search_batch_arrays(qs, 10, 12)
    r2 = ix.search_batch_arrays(qs, 10, 12)
    _assert_same(r1, r2)
    sel = rng.choice(3000, 100, replace=False)
    r3 = ix.search_batch_arrays(qs[sel], 10, 12)
    _assert_same((r1[0][sel], r1[1][sel], r1[2][sel]), r3)


def test_lists_many_lists_plan_without_lds_histogram(vh, oracle):
    """More lists (8,200) than the plan's LDS histogram holds (8,192 bins): the pair counting and
    scattering take their global-atomic path.  Checked against the query-major kernel and, exactly
    on integer parts, against the oracle."""
    rng = np.random.default_rng(93)
    parts = _skewed_parts(rng, 64, 8200, 30_000, integer=True)
    ix = _index(vh, parts, 64, 16, 256, vh.DistanceMetric.L2Squared)
    qs = rng.integers(-4, 5, (200, 64)).astype(np.float32)
    a, b = _both_paths(ix, qs, 10, 24)
    _assert_same(a, b)
    _check_search(vh, oracle, ix, parts, qs[:20], 10, 24, "l2", 16, 256, exact=True)


def test_batch_of_several_chunks(vh):
    """A batch whose (query, probe) pairs exceed one search chunk (2^22 pairs: 65,536 queries at
    nprobe 64) runs as several chunks; its results equal those of the same queries searched in
    batches of one chunk or less, bit for bit."""
    rng = np.random.default_rng(77)
    dim, nlist = 64, 64
    parts = _skewed_parts(rng, dim, nlist, 20_000)
    ix = _index(vh, parts, dim, 16, 256, vh.DistanceMetric.L2Squared)
    qs = rng.standard_normal((70_000, dim)).astype(np.float32)
    print("  70,000 queries at nprobe 64 (two chunks)", flush=True)
    whole = ix.search_batch_arrays(qs, 10, 64)
    head = ix.search_batch_arrays(qs[:40_000], 10, 64)
    tail = ix.search_batch_arrays(qs[40_000:], 10, 64)
    _assert_same(whole, tuple(np.concatenate([h, t]) for h, t in zip(head, tail)))


@pytest.mark.parametrize("metric", ["L2Squared", "DotProduct", "CosineSimilarity"])
@pytest.mark.parametrize("dim,k,nprobe,nq", [(32, 10, 8, 1024), (64, 1, 1, 1500), (128, 16, 64, 1100), (128, 10, 3, 2001),
                                             (64, 48, 16, 4100), (128, 10, 8, 1023)])
def test_eight_byte_rows_match_query_major(vh, metric, dim, k, nprobe, nq):
    """8-byte code rows at each sub-vector width, on both sides of the batch sizes that choose the path."""
    rng = np.random.default_rng(dim + 31 * k + nprobe)
    parts = _skewed_parts(rng, dim, 64, 50_000, empty=(5, 17, 40), m_sub=8)
    ix = _index(vh, parts, dim, 8, 256, vh.DistanceMetric[metric])
    a, b = _both_paths(ix, rng.standard_normal((nq, dim)).astype(np.float32), k, nprobe)
    _assert_same(a, b)


@pytest.mark.parametrize("m_sub,dim", [(16, 64), (16, 128), (8, 32), (8, 128)])
@pytest.mark.parametrize("metric", ["L2Squared", "CosineSimilarity"])
@pytest.mark.parametrize("empty", [(23,), (19, 20, 21, 22, 23), tuple(range(1, 24)), (0, 23)])
def test_last_lists_empty(vh, m_sub, dim, metric, empty):
    """No code row lies behind an empty last list, so its work items may load none: the last list
    empty, the last five, all but the first (one row in all), the first and the last."""
    rng = np.random.default_rng(dim + 100 * m_sub + len(empty))
    nlist = 24
    n = 1 if len(empty) == nlist - 1 else 3000
    parts = _skewed_parts(rng, dim, nlist, n, empty=empty, m_sub=m_sub)
    assert all(parts[2][c] == 0 for c in empty)
    ix = _index(vh, parts, dim, m_sub, 256, vh.DistanceMetric[metric])
    qs = rng.standard_normal((1100, dim)).astype(np.float32)
    for nprobe in (1, 24):
        a, b = _both_paths(ix, qs, 10, nprobe)
        _assert_same(a, b)
    assert np.all(a[2] == min(n, 10)), "every list was probed"


@pytest.mark.parametrize("nlist,n,k,nprobe,nq", [(64, 20_000, 10, 4, 1024), (64, 20_000, 10, 4, 1025), (64, 20_000, 10, 2, 1024),
                                                 (16, 40_000, 10, 8, 1024), (1500, 30_000, 10, 2, 1499),
                                                 (1500, 30_000, 10, 2, 1500), (2100, 30_000, 20, 3, 4199),
                                                 (2100, 30_000, 20, 3, 4200), (64, 10_000, 48, 21, 4096),
                                                 (64, 10_000, 48, 22, 4096)])
def test_eight_byte_rows_around_the_choice_of_path(vh, nlist, n, k, nprobe, nq):
    """Both sides of the batch sizes, list counts and k x nprobe at which 8-byte rows change paths."""
    rng = np.random.default_rng(nlist + nq)
    parts = _skewed_parts(rng, 64, nlist, n, m_sub=8)
    ix = _index(vh, parts, 64, 8, 256, vh.DistanceMetric.L2Squared)
    a, b = _both_paths(ix, rng.standard_normal((nq, 64)).astype(np.float32), k, nprobe)
    _assert_same(a, b)
