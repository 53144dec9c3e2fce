"""Spilled coarse rows (more than 4096 fine edges) of many and few members,
long and short ones, whose edges cross the gather's chunks, with counts of
coarse vertices around powers of two (the sort keys' widths), against the
oracle. Weights are sums of integers, so every array must be equal."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc", [2, 3, 64, 65, 1024, 1025])
@pytest.mark.parametrize("members", ["many", "few"])
def test_spilled_rows(nc, members):
    rs = np.random.default_rng(nc)
    n = 70000  # above the sizes a team contracts
    hubs = [6000, 5000, 4097, 4096, 1023, 1024, 1025, 9000]
    u = [np.full(d, h) for h, d in enumerate(hubs)]
    v = [len(hubs) + rs.permutation(n - len(hubs))[:d] for d in hubs]
    # short rows, isolated vertices among them
    u.append(rs.integers(len(hubs), n, 60000))
    v.append(rs.integers(len(hubs), n, 60000))
    u, v = np.concatenate(u), np.concatenate(v)
    key = np.unique(np.minimum(u, v).astype(np.int64) * n + np.maximum(u, v))
    u, v = key // n, key % n
    u, v = u[u != v], v[u != v]
    g = graphs.from_edges(n, u, v, rs.integers(1, 50, len(u)))
    if members == "many":
        mp = (rs.random(n) ** 3 * nc).astype(np.int32)  # a few aggregates of thousands of short rows
    else:
        mp = (np.arange(n) % nc).astype(np.int32)
    mp[:nc] = np.arange(nc)
    print("spill", nc, members, flush=True)
    got, exp = jet_amd.contract(g, mp, nc), oracle.contract(g, mp, nc)
    for k in ("rowptr", "col", "ew", "vw"):
        assert np.array_equal(got[k], exp[k]), k
