"""The order in which the row-per-lane scans (knn_rows.hip) run their workgroups: every pair of row group and
query tile exactly once, also where the queries are taken in several chunks (2 MB of queries each) and
where row groups leave places of the last XCDs idle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# Rows: filter rounds of 24 + 47 groups (spread, idle places at most 8%), 12 (plain) and 24 + 96 + ... (64 and
# more); queries: one chunk, a chunk and one tile more, and three chunks with the last one partial.
@pytest.mark.parametrize("metric", ["Manhattan", "Jaccard"])
@pytest.mark.parametrize("n,dim,nq", [(20_000, 1000, 512), (20_000, 1000, 528), (20_000, 993, 1411), (5000, 1000, 1100),
                                      (49_001, 480, 2100), (20_000, 24, 500)])
def test_query_chunks(metric, n, dim, nq):
    import vector_hip as vh

    rng = np.random.default_rng(nq)
    base = rng.uniform(-1, 1, (n, dim)).astype(np.float32)
    q = rng.uniform(-1, 1, (nq, dim)).astype(np.float32)
    eng = vh.CudaKnnEngine(base, dim, vh.DistanceMetric[metric])
    ids, dist, lens = eng.search_batch_arrays(q, 10)
    assert np.all(lens == 10)
    for s in range(0, nq, 130):  # pieces of one chunk, with the same scores bit for bit
        i2, d2, _ = eng.search_batch_arrays(q[s:s + 130], 10)
        np.testing.assert_array_equal(ids[s:s + 130], i2)
        np.testing.assert_array_equal(dist[s:s + 130], d2)
