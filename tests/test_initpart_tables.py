"""The host initial partition on graphs on both sides of the rule that chooses
between its gain heap and its key table (average degree n / 32), and on graphs
it coarsens first. Both pick the largest gain and the smallest id, so the
partitions are those the heap alone gave: pinned by their digests."""
import hashlib

import numpy as np
import pytest

import graphs
import oracle


def skewed(n, pairs, power, seed, wmax):
    rs = np.random.default_rng(seed)
    a = (rs.random(pairs) ** power * n).astype(int)
    b = (rs.random(pairs) ** power * n).astype(int)
    key = np.unique(np.minimum(a, b).astype(np.int64) * n + np.maximum(a, b))
    u, v = key // n, key % n
    keep = u != v
    u, v = u[keep], v[keep]
    g = graphs.from_edges(n, u, v, rs.integers(1, wmax + 1, len(u)))
    g["vw"] = rs.integers(1, 9, n).astype(np.int32)
    return g


@pytest.mark.parametrize(
    "n,deg,k,wmax,digest",
    [
        (868, 400, 64, 30, "2dbe85a2ca"),
        (1900, 190, 256, 9, "935e992a6b"),
        (512, 14, 64, 5, "ed33668773"),
        (300, 9, 3, 1, "712029a86e"),
        (1000, 32, 7, 4, "ce97d532ec"),
        (1000, 31, 7, 4, "62f1797f54"),
        (2500, 300, 9, 3, "6d91c814ff"),
        (40, 39, 5, 3, "e61ecfc61f"),
    ],
)
def test_table_and_heap_agree(n, deg, k, wmax, digest):
    g = skewed(n, n * deg // 2, 1.6, n + deg, wmax)
    assert hashlib.md5(oracle.initpart(g, k, 1.03, seed=7).tobytes()).hexdigest()[:10] == digest


@pytest.mark.parametrize(
    "n,pairs,k,digest", [(16555, 500000, 64, "2c112aef31"), (60000, 150000, 64, "2fec7c30b2"), (3000, 9000, 8, "0877bda438")]
)
def test_coarsened_first(n, pairs, k, digest):
    g = skewed(n, pairs, 2.5, n, 30)
    assert hashlib.md5(oracle.initpart(g, k, 1.03, seed=7).tobytes()).hexdigest()[:10] == digest
