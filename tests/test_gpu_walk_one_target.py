"""The walk that gives each target a wavefront (k_walk1: point queries of both
precisions, step walks of small mixed contexts) where its stack and its last
pass can go wrong: trees of one to a few nodes, around the 64 nodes of a pass,
a chain of single-child nodes down to two particles 2^-40 of the box apart,
theta = 0 (every cell opens, so the stack runs in its narrow mode), point
counts around the wavefront's and the block's targets, and points outside the
domain; against the oracle's walk."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_common import big_case, gpu_ctx, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu


def _check(case, parts, idx, q=0, prec=(G.POTG_FP64, G.POTG_MIXED)):
    sim = oracle_sim(case)
    sim.set_particles(parts)
    st = sim.state()
    sim.set_state(q, st["m"], 0, 0.0, 0)
    sim.build_tree()
    xyz = np.stack([parts["x"][idx], parts["y"][idx], parts["z"][idx]], 1)
    Eo, co = np.zeros((len(idx), 3)), np.zeros((len(idx), 3), np.uint32)
    for k, i in enumerate(idx):
        s = O.WalkStats()
        Eo[k] = sim.field_at(int(i), *xyz[k], 1, s)
        co[k] = (s.n_cell, s.n_leaf, s.n_open)
    scale = np.linalg.norm(Eo, axis=1)
    for p in prec:
        ctx = gpu_ctx(case, parts, precision=p, q=q)
        ctx.build_tree()
        E, c = ctx.field_at(0, xyz, exclude=idx, counts=True)
        rel = np.linalg.norm(E - Eo, axis=1) / np.where(scale > 0, scale, 1.0)
        if p == G.POTG_FP64:
            assert np.array_equal(c, co)
            assert rel.max() <= 1e-12, rel.max()
        else:
            # float32: positions carry 6e-8 R, MAC decisions may flip at the
            # threshold
            assert np.all(c == co, axis=1).mean() > 0.99
            assert np.median(rel) < 1e-5, np.median(rel)


@pytest.mark.parametrize("N", [3, 9, 64, 65, 66, 513])
@pytest.mark.parametrize("dipoles", [0, 1], ids=["monopole", "dipoles"])
def test_small_trees(N, dipoles):
    case = dict(big_case(N, seed=N), dipoles=dipoles)
    parts = oracle_sim(case).particles()
    _check(case, parts, np.arange(1, N, dtype=np.uint32), q=-4)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 31, 33, 4096])
def test_point_counts(n):
    case = dict(big_case(5001, seed=3), dipoles=1)
    parts = oracle_sim(case).particles()
    idx = np.random.default_rng(n).choice(np.arange(1, 5001), n, replace=False).astype(np.uint32)
    _check(case, parts, idx)


def test_theta_zero_meets_every_leaf():
    case = dict(big_case(4001, seed=5), theta=0.0)
    parts = oracle_sim(case).particles()
    _check(case, parts, np.arange(1, 4001, 13, dtype=np.uint32))


def test_deep_chain():
    """Two particles 2^-40 of the box apart: one child per node for 30
    levels (the float32 walk cannot tell the two apart: float64 only)."""
    case = big_case(2001, seed=6)
    parts = oracle_sim(case).particles()
    side = 2.0 * float(case["args"]["-r"]) * float(case["args"]["-m"])
    for f in ("x", "y", "z"):
        parts[f][7] = parts[f][8] + side * 2.0 ** -40 * (-1.0 if parts[f][8] > 0.5 * side else 1.0)
    _check(case, parts, np.arange(1, 2001, 3, dtype=np.uint32), prec=(G.POTG_FP64,))


def test_points_outside_the_domain():
    case = big_case(3001, seed=9)
    parts = oracle_sim(case).particles()
    sim = oracle_sim(case)
    sim.build_tree()
    R = float(case["args"]["-r"]) * float(case["args"]["-m"])
    pts = R + R * np.array([[3.0, 0.0, 0.0], [0.0, -50.0, 2.0], [1.5, 1.5, 1.5], [-1.2, 0.0, 0.3]])
    want = np.array([sim.phi_at(*p) for p in pts])
    ctx = gpu_ctx(case, parts)
    ctx.build_tree()
    got = ctx.phi_at(0, pts)
    # a few hundred terms of either sign, each to a few units of 2^-53
    mag = 1.6021766e-19 * 3001 / (4 * np.pi * 8.85419e-12) / np.linalg.norm(pts - R, axis=1)
    assert np.all(np.abs(got - want) <= 1e-12 * np.abs(want) + 1e-14 * mag)


def test_step_walk_of_a_small_context():
    """A small mixed context's step: targets, tallies and state as the float64
    path's, which walks 64 targets per wavefront."""
    case = dict(big_case(3003, seed=10), dipoles=1)
    parts = oracle_sim(case).particles()
    a = gpu_ctx(case, parts, precision=G.POTG_MIXED, seed=2)
    b = gpu_ctx(case, parts, precision=G.POTG_FP64, seed=2)
    oa, ob = a.step()[0], b.step()[0]
    assert oa == ob
    pa, pb = a.download(0)[0], b.download(0)[0]
    vs = np.abs(pb["vx"]).max()
    for f in ("vx", "vy", "vz"):
        # a step turns a velocity by about 1e-2 at most, the float32 field is
        # good to 2e-3 at its 99th percentile and 1e-5 at its median
        assert np.percentile(np.abs(pa[f] - pb[f]), 99) < 2e-5 * vs
        assert np.median(np.abs(pa[f] - pb[f])) < 1e-7 * vs
