"""Heavy edge coarsening of a level in one launch (levels of up to wg_max_n
vertices) against the oracle and the multi-kernel path: sizes around the
chunks and workgroups, equal weights, vertices too heavy to join, isolated
vertices, long rows and long chains of heavy neighbours. Maps are equal."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


def check(g, seed=3, level=1):
    for u in (False, True):
        em, enc = oracle.coarsen_map(g, 1, u, seed, level)
        for wg in (65536, 0):
            with jet_amd.tuned(wg_max_n=wg):
                m, nc = jet_amd.coarsen_map(g, 1, u, seed, level)
            assert nc == enc and np.array_equal(m, em), (u, wg)


@pytest.mark.parametrize("nx,ny", [(1, 1), (1, 2), (7, 9), (8, 8), (5, 13), (17, 15), (60, 70), (256, 256), (257, 256)])
@pytest.mark.parametrize("wmax", [1, 4, 1000])
def test_sizes(nx, ny, wmax):
    print("hec", nx, ny, wmax, flush=True)
    g = graphs.with_weights(graphs.grid2d(nx, ny), seed=nx, wmax=wmax)
    check(g)
    vw = np.ones(nx * ny, dtype=np.int32)
    vw[:: 7] = 50  # above six times the average in part of them
    g["vw"] = vw
    check(g)


@pytest.mark.parametrize("leaves", [3, 64, 513, 3000])
def test_stars_and_isolated(leaves):
    hubs = 8
    u = np.repeat(np.arange(hubs), leaves)
    v = hubs + np.arange(hubs * leaves)
    c = np.arange(hubs - 1)
    g = graphs.from_edges(hubs + hubs * leaves + 700, np.concatenate([u, c]), np.concatenate([v, c + 1]))
    print("stars", leaves, flush=True)
    check(g)


@pytest.mark.parametrize("n", [65, 5000, 40000])
def test_chains(n):
    # weights that grow along a path: every vertex's heavy neighbour is the
    # next one, a chain through all workgroups; shuffled ids
    rs = np.random.default_rng(n)
    ids = rs.permutation(n)
    for p in (np.arange(n), ids):
        g = graphs.from_edges(n, p[:-1], p[1:], np.arange(1, n))
        print("chain", n, flush=True)
        check(g)
