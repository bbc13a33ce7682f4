"""Keys and sort, through the tree they lead to, bit for bit against the
oracle's: particle counts around a tile's 1024 and around the sizes where the
passes' ways and the method change, batches whose grains' keys (the highest)
fill the ends of tiles, particles on the faces of cells and a hair beside them
(where the whole part of a scaled coordinate does not settle the digits), and
particles equal in every digit that a key holds, within a tile and across
tiles."""
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
    ctx = gpu_ctx(case, parts)
    ctx.build_tree()
    _equal(ctx.tree_canon(0), sim.tree_canon())


@pytest.mark.parametrize("N,geometry", [(1023, 0), (1024, 1), (1025, 0), (2049, 2), (4097, 0),
                                        (65536, 0), (65537, 0), (250000, 0), (250001, 0),
                                        (899999, 0), (900001, 0)])
def test_counts(N, geometry):
    case = big_case(N, geometry=geometry, A=(1.0, 2.0, 0.5)[geometry], seed=N)
    _check(case, oracle_sim(case).particles())


def test_batch_with_spheroid_grains():
    cases = [big_case(n, geometry=g, A=2.0 if g else 1.0, seed=n)
             for n, g in ((341, 1), (342, 1), (343, 0), (1024, 1), (2047, 1))]
    ctx = G.Context([gpu_config(c) for c in cases], G.POTG_FP64)
    sims = []
    for k, c in enumerate(cases):
        sims.append(oracle_sim(c))
        ctx.upload(k, sims[k].particles().view(G.PARTICLE_DT))
    ctx.build_tree()
    for k, sim in enumerate(sims):
        sim.build_tree()
        _equal(ctx.tree_canon(k), sim.tree_canon())


@pytest.mark.parametrize("bits", [5, 12, 21])
def test_on_the_faces(bits):
    N = 3001
    case = big_case(N, seed=bits)
    parts = oracle_sim(case).particles()
    side = 2.0 * float(case["args"]["-r"]) * float(case["args"]["-m"])
    rng = np.random.default_rng(bits)
    cells = np.unique(rng.integers(0, 1 << bits, (4 * N, 3)), axis=0)
    cells = cells[rng.permutation(len(cells))][:N - 1]
    x = side * cells / (1 << bits)
    # every third exactly on a face, the others an ulp below or above
    off = np.arange(N - 1) % 3
    for d, f in enumerate(("x", "y", "z")):
        v = np.where(off == 1, np.nextafter(x[:, d], side), x[:, d])
        v = np.where(off == 2, np.nextafter(v, 0.0), v)
        parts[f][1:] = v
    _check(case, parts)


@pytest.mark.parametrize("gap", [1, 1500])
def test_equal_keys(gap):
    # pairs and a run of five 2^-30 of the side apart: one key
    N = 4001
    case = big_case(N, seed=2)
    parts = oracle_sim(case).particles()
    side = 2.0 * float(case["args"]["-r"]) * float(case["args"]["-m"])
    for k in range(40):
        a, b = 100 + 3 * k, 100 + 3 * k + gap
        for f in ("x", "y", "z"):
            parts[f][b] = parts[f][a] + side * 2.0 ** -30
    for k in range(5):
        for f in ("x", "y", "z"):
            parts[f][3500 + k] = parts[f][3500] + k * side * 2.0 ** -32
    _check(case, parts)
