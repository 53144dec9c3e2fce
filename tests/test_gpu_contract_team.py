"""The one-launch contraction (k_contract_team) at the edges of its row sizes
(32 and 128 fine edges, 4 members, 2048 fine edges, above which the level goes
back to the general kernels) and of its teams, against the oracle. Weights are
sums of integers, so every array must be equal."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


def check(g, mp, nc):
    got, exp = jet_amd.contract(g, mp, nc), oracle.contract(g, mp, nc)
    for key in ("rowptr", "col", "ew", "vw"):
        assert np.array_equal(got[key], exp[key]), key


def stars(degrees, leaves, seed=2):
    rs = np.random.default_rng(seed)
    u = np.concatenate([np.full(d, h) for h, d in enumerate(degrees)])
    v = np.concatenate([len(degrees) + rs.permutation(leaves)[:d] for d in degrees])
    return graphs.from_edges(len(degrees) + leaves, u, v, rs.integers(1, 50, len(u)))


@pytest.mark.parametrize("longest", [2047, 2048, 2049])
@pytest.mark.parametrize("groups", [1, 7, 900, 3000])
def test_rows_at_table_edges(longest, groups):
    degrees = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 511, 513, 1024, longest]
    leaves = 3000
    g = stars(degrees, leaves)
    H = len(degrees)
    # the leaves of one group would be a row of all edges: leave them apart there
    lm = H + (np.arange(leaves) % groups if groups > 1 else np.arange(leaves))
    mp = np.concatenate([np.arange(H), lm]).astype(np.int32)
    print("tables", longest, groups, flush=True)
    check(g, mp, int(mp.max()) + 1)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1000, 4097, 65536])
@pytest.mark.parametrize("members", [1, 2, 3, 4, 5, 17])
def test_sizes_and_members(n, members):
    nx = max(1, int(np.sqrt(n)))
    ids = np.arange(n)
    u = np.concatenate([ids[:-1], ids[: max(0, n - nx)]])
    v = np.concatenate([ids[1:], ids[nx:] if n > nx else ids[:0]])
    rs = np.random.default_rng(n)
    g = graphs.from_edges(n, u, v, rs.integers(1, 9, len(u)))
    mp = (np.arange(n) // members).astype(np.int32)
    rs.shuffle(mp)
    print("members", n, members, flush=True)
    check(g, mp, int(mp.max()) + 1)


def test_coarse_rows_without_members():
    n = 2000
    g = graphs.from_edges(n, np.arange(n - 1), np.arange(1, n), np.ones(n - 1, dtype=np.int64))
    check(g, (3 * (np.arange(n) // 3)).astype(np.int32), n)


@pytest.mark.parametrize("n,nc", [(2048, 1), (2049, 1), (5000, 3), (30000, 64), (65536, 65), (65536, 1)])
def test_few_coarse_rows_of_many_vertices(n, nc):
    # hardly an edge: the fine vertices, not the rows, ask for workgroups
    rs = np.random.default_rng(n + nc)
    e = min(32 * nc, n // 2)
    u = rs.permutation(n)
    g = graphs.from_edges(n, u[:e], u[e : 2 * e], rs.integers(1, 9, e))
    mp = rs.integers(0, nc, n).astype(np.int32)
    print("few rows", n, nc, flush=True)
    check(g, mp, nc)
