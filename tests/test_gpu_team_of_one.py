"""Levels on both sides of the sizes up to which one workgroup refines a level
by itself (700 vertices, 7000 edges). Each level's refinement equals the
oracle's: record and partition."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(2, 1), (64, 300), (699, 3000), (700, 3499), (700, 3500), (700, 3501), (701, 3000)])
@pytest.mark.parametrize("k", [2, 9, 64])
def test_one_workgroup(n, m, k):
    rs = np.random.default_rng(n + m)
    ring = np.arange(n - 1)
    pairs = {(int(a), int(a) + 1) for a in ring}
    while len(pairs) < m:
        a, b = sorted(rs.integers(0, n, 2))
        if a != b:
            pairs.add((int(a), int(b)))
    u, v = np.array(sorted(pairs)).T
    g = graphs.from_edges(n, u, v, rs.integers(1, 9, len(u)))
    p0 = rs.integers(0, k, n).astype(np.int32)
    print("one", n, m, k, flush=True)
    p, rec = jet_amd.refine_level(g, p0, k, 1.05, uniform=False)
    ep, erec = oracle.refine_level(g, p0, k, 1.05, uniform=False)
    assert list(rec) == list(erec), (rec, erec)
    assert np.array_equal(p, ep)
