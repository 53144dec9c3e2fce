"""The update passes' slices of long moved rows (k_row_slices, k_update_big):
rows at the edges of the slice size and of the threshold, whose neighbours are
short rows, with few and many moves. Each level's refinement equals the
oracle's: record and partition."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [3, 64, 300])
@pytest.mark.parametrize("noise", [0.01, 1.0])
def test_long_rows_at_slice_edges(k, noise):
    # hubs joined to grid vertices of degree at most 4 + 14: no pulled rows but the hubs
    rs = np.random.default_rng(11)
    nx, ny = 330, 310
    n = nx * ny
    ids = np.arange(n).reshape(ny, nx)
    u = [ids[:, :-1].ravel(), ids[:-1, :].ravel()]
    v = [ids[:, 1:].ravel(), ids[1:, :].ravel()]
    degrees = [2047, 2048, 2049, 3071, 3072, 3073, 5000] * 2
    for h, d in enumerate(degrees):
        u.append(np.full(d, n + h))
        v.append(rs.choice(n, d, replace=False))
    u, v = np.concatenate(u), np.concatenate(v)
    g = graphs.from_edges(n + len(degrees), u, v, rs.integers(1, 9, len(u)))
    p0 = (np.arange(n + len(degrees)) * k // (n + len(degrees))).astype(np.int32)
    odd = rs.random(n + len(degrees)) < noise
    p0[odd] = rs.integers(0, k, int(odd.sum()))
    p0[n:] = 0  # every hub in one part: some of them move
    print("slices", k, noise, flush=True)
    p, rec = jet_amd.refine_level(g, p0, k, 1.03, uniform=False)
    ep, erec = oracle.refine_level(g, p0, k, 1.03, uniform=False)
    assert list(rec) == list(erec), (rec, erec)
    assert np.array_equal(p, ep)
