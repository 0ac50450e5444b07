"""The narrow resident-tile MFMA search kernel at row widths it takes (129 to 896 floats): every odd count of
32-float chunks, even ones, widths with padding, row ranges that end inside a 512-row stage and query
tiles that end inside 32 columns."""
import numpy as np
import pytest

from knn_check import check_knn

pytestmark = pytest.mark.gpu

NAMES = {"l2": "L2Squared", "dot": "DotProduct", "cosine": "CosineSimilarity"}


@pytest.mark.parametrize("metric", ["l2", "dot", "cosine"])
@pytest.mark.parametrize("dim", [129, 160, 191, 200, 288, 300, 352, 416, 420, 480, 500, 544, 545, 608, 672, 700,
                                 736, 800, 831, 864, 865, 896])
def test_row_widths(oracle, metric, dim):
    import vector_hip as vh

    rng = np.random.default_rng(dim)
    n = 9000 + dim
    base = rng.standard_normal((n, dim)).astype(np.float32)
    q = rng.standard_normal((141, dim)).astype(np.float32)
    ids, dist, lens = vh.CudaKnnEngine(base, dim, vh.DistanceMetric[NAMES[metric]]).search_batch_arrays(q, 10)
    assert np.all(lens == 10)
    # fp32 sums of dim terms of size about 1 (dot product: relative to the terms, not to their sum)
    check_knn(oracle, base, q, ids, dist, 10, metric, rtol=1e-4, atol=1e-4)
