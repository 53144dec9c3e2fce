"""Contraction at the edges of its row tiers (wave table, two workgroup table
sizes, radix spill) and with long runs of equal spill keys, against the
oracle. Weights are sums of integers, so every array must be equal."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu

DEGREES = [127, 128, 129, 1023, 1024, 1025, 2047, 4095, 4096, 4097, 9000]
LEAVES = 9000


def hub_graph():
    """One hub per entry of DEGREES, joined to that many distinct leaves."""
    rs = np.random.default_rng(3)
    u, v, w = [], [], []
    for h, d in enumerate(DEGREES):
        leaves = rs.permutation(LEAVES)[:d]
        u.append(np.full(d, h))
        v.append(len(DEGREES) + leaves)
        w.append(rs.integers(1, 50, d))
    return graphs.from_edges(len(DEGREES) + LEAVES, np.concatenate(u), np.concatenate(v), np.concatenate(w))


@pytest.mark.parametrize("groups", [LEAVES, LEAVES // 2, 700, 70, 3, 1])
@pytest.mark.parametrize("merge_hubs", [False, True])
def test_rows_at_tier_edges(groups, merge_hubs):
    g = hub_graph()
    H = len(DEGREES)
    hubs = np.arange(H) // (2 if merge_hubs else 1)
    leaves = hubs.max() + 1 + np.arange(LEAVES) % groups
    mp = np.concatenate([hubs, leaves]).astype(np.int32)
    nc = int(mp.max()) + 1
    print("tiers", groups, merge_hubs, nc, flush=True)
    got, exp = jet_amd.contract(g, mp, nc), oracle.contract(g, mp, nc)
    for key in ("rowptr", "col", "ew", "vw"):
        assert np.array_equal(got[key], exp[key]), key


def test_every_row_spills_or_vanishes():
    # everything in two aggregates (two spilled rows), then in one (a spilled
    # row without any edge)
    g = hub_graph()
    n = len(g["rowptr"]) - 1
    for nc in (2, 1):
        mp = (np.arange(n) % nc).astype(np.int32)
        got, exp = jet_amd.contract(g, mp, nc), oracle.contract(g, mp, nc)
        for key in ("rowptr", "col", "ew", "vw"):
            assert np.array_equal(got[key], exp[key]), (nc, key)
