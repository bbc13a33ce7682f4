"""The scans' tile sums where a launch of its own adds them up (65536 tiles of
1024: 68M particles in one context): every instance of a batch of equal ones has
the potential of one alone at the same points, pushes as many particles, and
ends a step in the same state, bit for bit.  A tile's offset that is off by any
number misplaces nodes, children or targets of some instance."""
import numpy as np
import pytest

from gpu_common import big_case, domain_radius, gpu_config, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu


def test_tile_sums_of_a_large_batch():
    N, n_inst = 400001, 170
    case = dict(big_case(N, seed=41), theta=0.9)
    parts = oracle_sim(case).particles().view(G.PARTICLE_DT)
    cfg = gpu_config(case, 5)
    batch, one = G.Context([cfg] * n_inst, G.POTG_MIXED), G.Context([cfg], G.POTG_MIXED)
    for c in (batch, one):
        c.set_tuning(2048, 64, 1)
        for k in range(c.n_inst):
            c.upload(k, parts, q=-30)
        c.build_tree()
    R = domain_radius(case)
    pts = R + 0.9 * R * np.random.default_rng(1).uniform(-1.0, 1.0, (64, 3))
    phi = one.phi_at(0, pts)
    for k in range(n_inst):
        assert np.array_equal(batch.phi_at(k, pts), phi), k
    want = one.step()[0]
    p1, g1 = one.download(0)
    assert all(o == want for o in batch.step())
    for k in (0, 1, 84, 168, 169):
        p, g = batch.download(k)
        assert np.array_equal(p.view(np.uint8), p1.view(np.uint8)) and g == g1, k
