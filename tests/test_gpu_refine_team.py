"""Levels refined in one launch by a team of workgroups (wg_max_n) at the
edges of its ranges: vertices per workgroup and chunk, the number of parts its
LDS holds, rows around the sixteen lanes that build them, steps that rebuild
tables, long re-draw lists, and calls from several threads at once. Every
record and partition equals the oracle's."""
import threading

import numpy as np
import pytest

import graphs
import jet_amd
import oracle
from test_refsim_refine import rand_part

pytestmark = pytest.mark.gpu


def check(g, p0, k, imb, **kw):
    p, rec = jet_amd.refine_level(g, p0, k, imb, uniform=g["uniform"], **kw)
    ep, erec = oracle.refine_level(g, p0, k, imb, uniform=g["uniform"], **kw)
    assert list(rec) == list(erec), (rec, erec)
    assert np.array_equal(p, ep)


# 1024 / 8192: team sizes change; 64 per chunk; 65,536 the largest level
@pytest.mark.parametrize("nx,ny", [(1, 1), (1, 2), (7, 9), (8, 8), (5, 13), (31, 33), (32, 32), (41, 25), (64, 128),
                                   (83, 99), (256, 256), (257, 255)])
@pytest.mark.parametrize("skew", [0.0, 1.5])
def test_level_sizes(nx, ny, skew):
    g = graphs.with_weights(graphs.grid2d(nx, ny), seed=nx, wmax=5, vwmax=3) if nx * ny > 1 else graphs.path(1)
    n = nx * ny
    k = min(8, n)
    print("sizes", nx, ny, skew, flush=True)
    check(g, rand_part(n, k, 4, skew) if n > 1 else np.zeros(1, np.int32), k, 1.03)


@pytest.mark.parametrize("k", [1, 2, 63, 64, 65, 255, 256, 257])
def test_part_counts(k):
    g = graphs.with_weights(graphs.random_graph(3000, 30000, seed=2), seed=3, wmax=7, vwmax=4)
    print("parts", k, flush=True)
    check(g, rand_part(3000, k, 5, 1.0), k, 1.05)


def test_row_lengths_around_the_build_tiers():
    rs = np.random.default_rng(8)
    u, v = [], []
    n = 2500
    for h, d in enumerate([15, 16, 17, 31, 33, 63, 64, 65, 200, 1000] * 3):
        u.append(np.full(d, h))
        v.append(100 + rs.choice(n - 100, d, replace=False))
    u.append(np.arange(100, n - 1))
    v.append(np.arange(101, n))
    g = graphs.from_edges(n, np.concatenate(u), np.concatenate(v), rs.integers(1, 9, sum(len(x) for x in u)))
    for k in (3, 16, 100):
        print("rows", k, flush=True)
        check(g, rand_part(n, k, 6, 0.5), k, 1.04)


def test_isolated_vertices_and_empty_rows():
    g = graphs.from_edges(500, np.arange(100), np.arange(1, 101))
    check(g, rand_part(500, 5, 3, 1.0), 5, 1.02)


@pytest.mark.parametrize("longest", [128, 129, 700])
def test_many_edges_with_and_without_long_rows(longest):
    # above 100,000 edges the team declines levels with longer rows than 128;
    # the multi-kernel path takes them
    g = graphs.random_graph(8000, 60000, seed=4, wmax=6)
    u = np.repeat(np.arange(8000), np.diff(g["rowptr"]))
    keep = u < g["col"]
    extra = 100 + np.random.default_rng(2).choice(7900, longest, replace=False)
    row0 = (u != 0) & (g["col"] != 0) & keep
    uu = np.concatenate([u[row0], np.zeros(longest, np.int64)])
    vv = np.concatenate([g["col"][row0], extra])
    g = graphs.from_edges(8000, uu, vv, np.concatenate([g["ew"][row0], np.full(longest, 2)]))
    assert len(g["col"]) > 100000 and np.diff(g["rowptr"]).max() == longest
    for k, skew in ((4, 1.0), (32, 0.3)):
        print("edges", longest, k, flush=True)
        check(g, rand_part(8000, k, 8, skew), k, 1.03)


def test_heavy_vertices_redraw():
    # few heavy vertices in one part: strong steps with more re-draws than the
    # LDS list holds
    g = graphs.with_weights(graphs.grid2d(120, 90), seed=1, wmax=3, vwmax=60)
    n = 120 * 90
    p0 = np.zeros(n, np.int32)
    p0[: n // 50] = np.arange(n // 50) % 64
    check(g, p0, 64, 1.01)


def test_concurrent_calls():
    g = graphs.with_weights(graphs.grid2d(70, 60), seed=9, wmax=4)
    cfg = jet_amd.Config(num_parts=12, max_imb_ratio=1.03, coarsening_alg=0)
    ref, cut = jet_amd.partition_csr(g, cfg, seed=3)
    epart, ecut, _ = oracle.partition(g, 12, 1.03, alg=0, seed=3)
    assert cut == ecut and np.array_equal(ref, epart)
    bad = []

    def work(ctx):
        for t in [ctx.submit(g, cfg, seed=3) for _ in range(6)]:
            part, c, _, _ = ctx.poll(t)
            if c != cut or not np.array_equal(part, ref):
                bad.append(c)

    with jet_amd.Context(workers=5) as a, jet_amd.Context(workers=12) as b:
        ts = [threading.Thread(target=work, args=(x,)) for x in (a, b)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    assert not bad
