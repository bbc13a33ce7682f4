"""The tree's nodes, bit for bit against the oracle's, at the sizes where the
pass that computes the moments can go wrong: trees of one node and around a
block's 256 nodes, around the sizes where its lists are taken by one block, by
groups of blocks and where the levels get a launch each, particles in close
pairs (more nodes, and so more and longer lists, than a block has lanes or LDS
slots for), a clump of deep cells, coordinates that are zero or subnormal, and
batches of trees of no particles, one and many."""
import numpy as np
import pytest

from gpu_common import big_case, gpu_config, gpu_ctx, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu


def _equal(got, ref):
    for f in ("depth", "is_leaf", "q", "aq", "nchild", "c"):
        assert np.array_equal(got[f], ref[f]), f
    leaf = ref["is_leaf"] == 1
    assert np.array_equal(got["part"][leaf], ref["part"][leaf])


def _check(case, parts):
    sim = oracle_sim(case)
    sim.set_particles(parts)
    sim.build_tree()
    ref = sim.tree_canon()
    ctx = gpu_ctx(case, parts)
    ctx.build_tree()
    got = ctx.tree_canon(0)
    _equal(got, ref)
    if case.get("dipoles"):
        assert np.array_equal(ctx.tree_dipoles(0), sim.tree_dipoles())


@pytest.mark.parametrize("N", [3, 9, 470, 520, 570, 2111, 20447, 20449, 70001, 599999, 600001])
@pytest.mark.parametrize("dipoles", [0, 1], ids=["monopole", "dipoles"])
def test_sizes(N, dipoles):
    case = dict(big_case(N, seed=N), dipoles=dipoles)
    _check(case, oracle_sim(case).particles())


@pytest.mark.parametrize("N,share", [(20001, 0.12), (60001, 0.12), (20001, 0.5)])
@pytest.mark.parametrize("dipoles", [0, 1], ids=["monopole", "dipoles"])
def test_close_pairs(N, share, dipoles):
    case = dict(big_case(N, seed=7), dipoles=dipoles)
    parts = oracle_sim(case).particles()
    R = float(case["args"]["-r"]) * float(case["args"]["-m"])
    sep = share * R * N ** (-1.0 / 3.0)
    for f in ("x", "y", "z"):
        parts[f][2::2] = parts[f][1:-1:2] + np.where(parts[f][1:-1:2] > R, -sep, sep)
    _check(case, parts)


def test_deep_clump():
    # cells halved some 45 times, and coordinates next to zero
    case = dict(big_case(3001, seed=5), dipoles=1)
    parts = oracle_sim(case).particles()
    R = float(case["args"]["-r"]) * float(case["args"]["-m"])
    rng = np.random.default_rng(3)
    for f in ("x", "y", "z"):
        parts[f][100:120] = R * (1.0 + rng.random(20) * 2.0 ** -35)
    parts["y"][200] = 0.0
    parts["z"][201] = 1e-310
    parts["x"][202] = 1e-280
    _check(case, parts)


def test_batch_of_bare_trees():
    # a spheroid grain is not in the tree: particles 1 of 2, 2 of 3
    cases = [big_case(n, geometry=g, A=2.0 if g else 1.0, seed=n)
             for n, g in ((3, 1), (3, 0), (700, 0), (4, 1))]
    parts = [oracle_sim(c).particles() for c in cases]
    ctx = G.Context([gpu_config(c) for c in cases], G.POTG_FP64)
    for k, p in enumerate(parts):
        ctx.upload(k, p.view(G.PARTICLE_DT))
    ctx.build_tree()
    for k, c in enumerate(cases):
        sim = oracle_sim(c)
        sim.build_tree()
        ref, got = sim.tree_canon(), ctx.tree_canon(k)
        _equal(got, ref)


@pytest.mark.parametrize("n_inst,N", [(16, 37600), (40, 15100), (1100, 550)])
def test_large_batches(n_inst, N):
    # more tree particles than the blocks of nodes take: level by level, the
    # top levels' nodes shared out by the number of trees
    case = big_case(N, seed=n_inst)
    sim = oracle_sim(case)
    parts = sim.particles().view(G.PARTICLE_DT)
    sim.build_tree()
    ref = sim.tree_canon()
    ctx = G.Context([gpu_config(case)] * n_inst, G.POTG_FP64)
    for k in range(n_inst):
        ctx.upload(k, parts)
    ctx.build_tree()
    for k in (0, 1, n_inst // 2, n_inst - 1):
        _equal(ctx.tree_canon(k), ref)
