"""Teams that do not gather: with team_start_spins = 0 the first workgroup of
every team gives up at once, every workgroup ends, and matching, contraction and
refinement take the kernels of larger levels. Results equal the oracle's (whole
numbers: equality)."""
import numpy as np
import pytest

import graphs
import jet_amd
import oracle

pytestmark = pytest.mark.gpu

# just above one workgroup, ordinary, the largest a team takes
SIZES = [(33, 32), (150, 140), (256, 256)]


def grid(nx, ny):
    return graphs.with_weights(graphs.grid2d(nx, ny), seed=nx, wmax=4)


@pytest.mark.parametrize("alg", [0, 2])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_matching(nx, ny, alg):
    g = grid(nx, ny)
    em, enc = oracle.coarsen_map(g, alg, False, 3, 1)
    print("abandoned matching", nx, ny, alg, flush=True)
    with jet_amd.tuned(team_start_spins=0):
        m, nc = jet_amd.coarsen_map(g, alg, False, 3, 1)
    assert nc == enc and np.array_equal(m, em)


@pytest.mark.parametrize("nx,ny", SIZES)
def test_contraction(nx, ny):
    g = grid(nx, ny)
    mp, nc = oracle.coarsen_map(g, 0, False, 3, 1)
    exp = oracle.contract(g, mp, nc)
    print("abandoned contraction", nx, ny, flush=True)
    with jet_amd.tuned(team_start_spins=0):
        got = jet_amd.contract(g, mp, nc)
    for key in ("rowptr", "col", "ew", "vw"):
        assert np.array_equal(got[key], exp[key]), key


@pytest.mark.parametrize("nx,ny", SIZES)
def test_refinement(nx, ny):
    g = grid(nx, ny)
    p0 = np.random.default_rng(nx).integers(0, 8, nx * ny).astype(np.int32)
    ep, erec = oracle.refine_level(g, p0, 8, 1.03, uniform=False)
    print("abandoned refinement", nx, ny, flush=True)
    with jet_amd.tuned(team_start_spins=0):
        p, rec = jet_amd.refine_level(g, p0, 8, 1.03, uniform=False)
    assert list(rec) == list(erec) and np.array_equal(p, ep)


def test_call_after_an_abandoned_one_is_the_same():
    # a whole partition whose first team is given up, and one after it
    g = grid(150, 140)
    cfg = jet_amd.Config(num_parts=8, max_imb_ratio=1.03, coarsening_alg=0)
    ep, ec, _ = oracle.partition(g, 8, 1.03, alg=0, seed=5)
    for spins in (0, 1 << 18):
        print("partition", spins, flush=True)
        with jet_amd.tuned(team_start_spins=spins):
            p, c = jet_amd.partition_csr(g, cfg, seed=5)
        assert c == ec and np.array_equal(p, ep)


def test_batch_with_abandoned_teams():
    jobs = [grid(20 + 3 * i, 50 + i) for i in range(24)]
    cfgs = [jet_amd.Config(num_parts=4 + i % 5, coarsening_alg=i % 3) for i in range(24)]
    alone = [jet_amd.partition_csr(g, c, seed=i) for i, (g, c) in enumerate(zip(jobs, cfgs))]
    print("batch of 24, 16 workers", flush=True)
    with jet_amd.tuned(team_start_spins=0), jet_amd.Context(workers=16) as ctx:
        parts, cuts = ctx.batch(jobs, cfgs, list(range(24)))
    for i, (p, c) in enumerate(alone):
        assert cuts[i] == c and np.array_equal(parts[i], p), i
