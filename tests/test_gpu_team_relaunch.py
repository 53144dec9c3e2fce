"""A level whose iterations take several launches of the team (team_launch_iters)
against the oracle: a launch ends after every iteration, or after five, with the
step's best state kept, update_large's rows rebuilt and a rebalancing sequence
cut anywhere. Whole numbers: equality."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iters", [1, 5])
@pytest.mark.parametrize("name,mk,k", [
    ("one workgroup", lambda: graphs.with_weights(graphs.grid2d(23, 21), seed=1, wmax=4, vwmax=3), 4),
    ("eight", lambda: graphs.with_weights(graphs.grid2d(31, 30), seed=2, wmax=4, vwmax=3), 8),
    ("long rows", lambda: graphs.with_weights(graphs.rmat(11, 8, seed=7), seed=2, wmax=5), 16),
    ("thirty-two", lambda: graphs.with_weights(graphs.grid2d(110, 100), seed=4, wmax=3), 6),
])
def test_level_in_several_launches(name, mk, k, iters):
    g = mk()
    n = len(g["rowptr"]) - 1
    rs = np.random.default_rng(n)
    for skewed in (False, True):
        p0 = rs.integers(0, k, n).astype(np.int32)
        if skewed:
            p0[rs.random(n) < 0.7] = 0
        ep, erec = oracle.refine_level(g, p0, k, 1.03, uniform=False)
        print(name, iters, skewed, flush=True)
        with jet_amd.tuned(team_launch_iters=iters):
            p, rec = jet_amd.refine_level(g, p0, k, 1.03, uniform=False)
        assert list(rec) == list(erec) and np.array_equal(p, ep)
