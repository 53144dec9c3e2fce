"""What a job takes of the device against the estimate its admission uses (128 n
+ 48 m + 1 MiB). A context has two arenas, for the hierarchy and for scratch,
whose largest extents need not come at the same time; each new chunk is as large
as those before it together, so an arena reserves at most twice its extent and a
first chunk of 64 MiB."""
import ctypes

import numpy as np
import pytest

import graphs
import jet_amd

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert jet_amd.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_device_coarsening_of_long_rows_among_many_vertices():
    # 512 hubs of 4,200 neighbours, too heavy to merge, among 500,000 leaves:
    # weighted HEC keeps every vertex, and each hub's row is built with arrays
    # over all coarse vertices
    rs = np.random.default_rng(5)
    hubs, leaves, d = 512, 500000, 4200
    u = np.repeat(np.arange(hubs), d)
    v = hubs + np.concatenate([rs.choice(leaves, d, replace=False) for _ in range(hubs)])
    g = graphs.from_edges(hubs + leaves, u, v, rs.integers(1, 9, len(u)))
    g["vw"][:hubs] = 1000
    n, m = len(g["rowptr"]) - 1, len(g["col"])
    estimate = 128 * n + 48 * m + (1 << 20)
    with jet_amd.Context(workers=1) as ctx:
        free = free_bytes()
        print("hubs among leaves", n, m, flush=True)
        part, cut, _, _ = ctx.poll(ctx.submit(g, jet_amd.Config(num_parts=8, max_imb_ratio=1.1, coarsening_alg=1), seed=3))
        used = free - free_bytes()
    assert part.min() >= 0 and part.max() < 8
    print("used", used, "estimate", estimate, flush=True)
    assert used <= 2 * (2 * estimate + (64 << 20))
