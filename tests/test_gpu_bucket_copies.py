"""Rebalancing of large levels with few parts, whose bucket sums are kept in
several copies (one per 32 to 256 workgroups of the select kernels). Each
level's refinement equals the oracle's: record and partition."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(270, 260), (410, 350)])
@pytest.mark.parametrize("k", [2, 3, 4, 17, 64, 65])
def test_few_parts(nx, ny, k):
    g = graphs.with_weights(graphs.grid2d(nx, ny), seed=k, wmax=5)
    n = nx * ny
    rs = np.random.default_rng(k)
    # part 0 far too large: weak, then strong steps move much
    p0 = np.minimum(np.arange(n) * 2 * k // n, k - 1).astype(np.int32)[::-1].copy()
    odd = rs.random(n) < 0.02
    p0[odd] = rs.integers(0, k, int(odd.sum()))
    print("copies", n, k, flush=True)
    p, rec = jet_amd.refine_level(g, p0, k, 1.01, uniform=False)
    ep, erec = oracle.refine_level(g, p0, k, 1.01, uniform=False)
    assert list(rec) == list(erec), (rec, erec)
    assert np.array_equal(p, ep)
