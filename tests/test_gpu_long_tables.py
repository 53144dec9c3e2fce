"""Connectivity tables read by whole waves in the select kernels of large
levels: table sizes around 16 and 64 slots and the wave's multiples, few and
many vertices to evaluate. Each level's refinement equals the oracle's: record
and partition."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,k", [(700, 600, 40), (760, 700, 300)])
@pytest.mark.parametrize("noise", [0.001, 0.2])
def test_table_sizes(nx, ny, k, noise):
    rs = np.random.default_rng(nx)
    n = nx * ny
    ids = np.arange(n).reshape(ny, nx)
    u = [ids[:, :-1].ravel(), ids[:-1, :].ravel()]
    v = [ids[:, 1:].ravel(), ids[1:, :].ravel()]
    degrees = [11, 12, 13, 15, 16, 17, 18, 31, 33, 63, 64, 65, 127, 129, 255, 300, 700] * 40
    for h, d in enumerate(degrees):
        u.append(np.full(d, n + h))
        v.append(rs.integers(0, n, d))
    u, v = np.concatenate(u), np.concatenate(v)
    key = np.unique(u.astype(np.int64) * (n + len(degrees)) + v)
    u, v = key // (n + len(degrees)), key % (n + len(degrees))
    g = graphs.from_edges(n + len(degrees), u, v, rs.integers(1, 9, len(u)))
    N = n + len(degrees)
    p0 = (np.arange(N) * k // N).astype(np.int32)
    odd = rs.random(N) < noise
    p0[odd] = rs.integers(0, k, int(odd.sum()))
    # hubs start in a few oversized parts: the rebalancers evaluate them
    p0[n:] = rs.integers(0, 3, len(degrees))
    print("tables", N, k, noise, flush=True)
    p, rec = jet_amd.refine_level(g, p0, k, 1.02, uniform=False)
    ep, erec = oracle.refine_level(g, p0, k, 1.02, uniform=False)
    assert list(rec) == list(erec), (rec, erec)
    assert np.array_equal(p, ep)
