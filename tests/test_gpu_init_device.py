"""Partitions whose coarsest graph is large enough (2^21 adjacency entries) to be
coarsened on the device for the initial partition, against the oracle, which
does it on the host: partition, cut and level records. Rows of every tier of
the device's row builder (a wave, two workgroup sizes, dense arrays), long
proposers, heavy vertices that the weight cap keeps single, isolated vertices
and leaves of one hub."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


def run(g, k, imb, seed):
    cfg = jet_amd.Config(num_parts=k, max_imb_ratio=imb, coarsening_alg=1)
    part, cut, st = jet_amd.partition_csr(g, cfg, seed=seed, stats=True)
    epart, ecut, levels = oracle.partition(g, k, imb, alg=1, seed=seed, repeat_shortcut=True)
    assert cut == ecut
    assert np.array_equal(part, epart)
    assert [st.levels[i].total_iterations for i in range(st.num_levels)] == [x[4] for x in levels]


@pytest.mark.parametrize("leaf_pairs,seed", [(False, 5), (True, 6)])
def test_hub_and_leaf_fixed_point(leaf_pairs, seed):
    g = graphs.heavy_bipartite(60, 24000, seed=seed, density=0.9, leaf_pairs=leaf_pairs)
    assert len(g["col"]) >= 1 << 21
    print("hub and leaf", leaf_pairs, flush=True)
    run(g, 32, 1.05, seed)


def test_rows_of_every_tier():
    # hubs of 300 to 14,000 neighbours among leaves of about 200, hubs too
    # heavy to merge: weighted HEC keeps every vertex, so this is the coarsest
    # graph; some leaves have one neighbour or none
    rs = np.random.default_rng(3)
    leaves, hubs = 14000, 160
    size = np.unique(np.geomspace(300, 14000, hubs).astype(int))
    u, v = [], []
    for h, d in enumerate(size):
        u.append(np.full(d, h))
        v.append(len(size) + rs.permutation(leaves)[:d])
    u, v = np.concatenate(u), np.concatenate(v)
    n = len(size) + leaves + 500
    g = graphs.from_edges(n, u, v, rs.integers(1, 9, len(u)))
    g["vw"] = np.ones(n, np.int32)
    g["vw"][: len(size)] = 1000
    print("tiers", len(g["col"]), flush=True)
    cfg = jet_amd.Config(num_parts=16, max_imb_ratio=1.1, coarsening_alg=1)
    part, cut = jet_amd.partition_csr(g, cfg, seed=2)
    epart, ecut, _ = oracle.partition(g, 16, 1.1, alg=1, seed=2, repeat_shortcut=True)
    assert cut == ecut and np.array_equal(part, epart)


def test_irregular_graph():
    g = graphs.with_weights(graphs.rmat(17, 16, seed=9), seed=1, wmax=4)
    for seed in (1, 2):
        cfg = jet_amd.Config(num_parts=64, max_imb_ratio=1.1, coarsening_alg=1)
        part, cut = jet_amd.partition_csr(g, cfg, seed=seed)
        epart, ecut, _ = oracle.partition(g, 64, 1.1, alg=1, seed=seed, repeat_shortcut=True)
        assert cut == ecut and np.array_equal(part, epart)
