"""The scan of rows of degree above 64 for moved neighbours (k_pull_hubs): rows
at the edges of its chunk and tier sizes, few and many moves (flagged rows,
every row, tables rebuilt), part counts that change the waves per workgroup,
and a level whose vertices do not fit its bit array. Each level's refinement
equals the oracle's: record and partition."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


def hubs_on_grid(nx, ny, degrees, seed=1):
    """A grid plus one hub per entry of degrees, joined to that many of the
    grid's vertices; random weights."""
    rs = np.random.default_rng(seed)
    n = nx * ny
    ids = np.arange(n).reshape(ny, nx)
    u = [ids[:, :-1].ravel(), ids[:-1, :].ravel()]
    v = [ids[:, 1:].ravel(), ids[1:, :].ravel()]
    for h, d in enumerate(degrees):
        u.append(np.full(d, n + h))
        v.append(rs.choice(n, d, replace=False))
    u, v = np.concatenate(u), np.concatenate(v)
    return graphs.from_edges(n + len(degrees), u, v, rs.integers(1, 9, len(u)))


def check(g, p0, k, imb):
    p, rec = jet_amd.refine_level(g, p0, k, imb, uniform=False)
    ep, erec = oracle.refine_level(g, p0, k, imb, uniform=False)
    assert list(rec) == list(erec), (rec, erec)
    assert np.array_equal(p, ep)


@pytest.mark.parametrize("k", [2, 17, 600, 1100])
@pytest.mark.parametrize("noise", [0.002, 0.05, 1.0])
def test_rows_at_chunk_and_tier_edges(k, noise):
    degrees = [63, 64, 65, 66, 255, 256, 257, 511, 513, 2047, 2048, 2049, 5000] * 2
    g = hubs_on_grid(110, 100, degrees)
    n = len(g["rowptr"]) - 1
    rs = np.random.default_rng(5)
    p0 = (np.arange(n) * k // n).astype(np.int32)
    odd = rs.random(n) < noise
    p0[odd] = rs.integers(0, k, int(odd.sum()))
    print("edges", k, noise, flush=True)
    check(g, p0, k, 1.05)


@pytest.mark.parametrize("noise", [0.0005, 0.02])
def test_more_vertices_than_the_bits_hold(noise):
    # 56 KB of bits hold 458,752 vertices: here a bit stands for two
    k = 512
    g = hubs_on_grid(880, 830, [100, 3000, 40000] * 4)
    n = len(g["rowptr"]) - 1
    assert n > 458752
    rs = np.random.default_rng(6)
    p0 = (np.arange(n) * k // n).astype(np.int32)
    odd = rs.random(n) < noise
    p0[odd] = rs.integers(0, k, int(odd.sum()))
    print("stamps", noise, n, flush=True)
    check(g, p0, k, 1.05)
