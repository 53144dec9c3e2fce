"""The partition quality report with its per-part sums in LDS (up to 2048
parts) and in memory (above), against sums over the edges."""
import numpy as np
import pytest

import graphs
import jet_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 2, 2047, 2048, 2049, 3000])
def test_quality_sums(k):
    rs = np.random.default_rng(k)
    n = 9000
    u, v = rs.integers(0, n, 40000), rs.integers(0, n, 40000)
    key = np.unique(np.minimum(u, v).astype(np.int64) * n + np.maximum(u, v))
    u, v = key // n, key % n
    u, v = u[u != v], v[u != v]
    g = graphs.from_edges(n, u, v, rs.integers(1, 9, len(u)))
    part = rs.integers(0, k, n).astype(np.int32)
    part[:k] = np.arange(k)
    q = jet_amd.partition_quality(g, part, k)
    src = np.repeat(np.arange(n), np.diff(g["rowptr"]))
    cross = part[src] != part[g["col"]]
    per_part = np.bincount(part[src][cross], weights=np.asarray(g["ew"])[cross], minlength=k)
    pairs = np.unique(src[cross].astype(np.int64) * k + part[g["col"]][cross])
    assert (q.edge_cut, q.comm_size) == (int(per_part.sum()) // 2, len(pairs))
    assert q.max_part_cut == int(per_part.max())
