"""Matching of a level in one launch (levels of up to wg_max_n vertices) against
the oracle and the multi-kernel path: sizes around the chunks and workgroups,
2-hop groups around the size that is compared one by one, isolated vertices,
stars, twins, long rows. Maps are equal."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


def check(g, uniform=None, seeds=(0, 5), algs=(0, 2), level=1):
    for alg in algs:
        for u in ((False, True) if uniform is None else (uniform,)):
            for seed in seeds:
                em, enc = oracle.coarsen_map(g, alg, u, seed, level)
                for wg in (65536, 0):
                    with jet_amd.tuned(wg_max_n=wg):
                        m, nc = jet_amd.coarsen_map(g, alg, u, seed, level)
                    assert nc == enc and np.array_equal(m, em), (alg, u, seed, wg)


@pytest.mark.parametrize("nx,ny", [(1, 2), (7, 9), (8, 8), (5, 13), (16, 16), (17, 15), (60, 70), (256, 255),
                                   (256, 256), (257, 256)])
def test_sizes(nx, ny):
    print("sizes", nx, ny, flush=True)
    check(graphs.with_weights(graphs.grid2d(nx, ny), seed=nx, wmax=4), seeds=(3,))


def stars(hubs, leaves, extra=0):
    u = np.repeat(np.arange(hubs), leaves)
    v = hubs + np.arange(hubs * leaves)
    c = np.arange(hubs - 1)
    return graphs.from_edges(hubs + hubs * leaves + extra, np.concatenate([u, c]), np.concatenate([v, c + 1]))


@pytest.mark.parametrize("leaves", [1, 2, 3, 64, 65, 511, 512, 513, 514, 1500])
def test_leaf_groups(leaves):
    print("leaves", leaves, flush=True)
    check(stars(8, leaves), seeds=(1,))


@pytest.mark.parametrize("extra", [1, 2, 63, 512, 513, 700, 20001])
def test_isolated_vertices_are_twins(extra):
    print("isolated", extra, flush=True)
    check(stars(4, 40, extra), seeds=(1,), algs=(0,))


def test_twins_and_relatives():
    # complete bipartite blocks: the leaves of a block are twins of degree 3;
    # weighted, with hub degrees that differ by block
    rs = np.random.default_rng(4)
    u, v, w = [], [], []
    n = 0
    for size in (2, 5, 33, 600, 1100):
        h = n + np.arange(3)
        leaf = n + 3 + np.arange(size)
        u.append(np.repeat(h, size))
        v.append(np.tile(leaf, 3))
        w.append(rs.integers(1, 4, 3 * size))
        n += 3 + size
    u, v = np.concatenate(u), np.concatenate(v)
    # drop some edges: relatives instead of twins
    keep = rs.random(len(u)) < 0.8
    for k in (np.ones(len(u), bool), keep):
        print("twins", int(k.sum()), flush=True)
        check(graphs.from_edges(n, u[k], v[k], np.concatenate(w)[k]), seeds=(2,))


@pytest.mark.parametrize("scale,ef", [(9, 4), (12, 8), (14, 8), (16, 6)])
def test_irregular(scale, ef):
    print("rmat", scale, flush=True)
    check(graphs.with_weights(graphs.rmat(scale, ef, seed=scale), seed=2, wmax=5), seeds=(7,))


def test_edgeless():
    g = graphs.path(1)
    check(g, seeds=(0,))
    g = {"rowptr": np.zeros(301, np.int64), "col": np.zeros(0, np.int32), "ew": np.zeros(0, np.int32),
         "vw": np.ones(300, np.int32), "uniform": True}
    check(g, seeds=(0,))
