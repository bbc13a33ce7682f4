"""The float64 walk whose tiles are shared by four wavefronts, each taking a
part of the cells two levels below the root, at sizes and opening angles that
select it: uniform trees, a tree that is a chain of single children down to a
clump (every target's work in one part) with a few particles elsewhere, and a
batch with an instance of another kind.  The velocities a step gives its
electrons against the field that point queries -- one target a wavefront,
itself checked against the oracle -- return at the same half-drifted
positions, with the same interaction counts.

Tolerance: without a magnetic field a step turns v into v + dt q E / m exactly
but for a few roundings of float64 (2^-53 of |v| + |dv| each), and the two
walks sum the same terms in different orders: 1e-11 of |dv|, or, where a
target's terms cancel, of the median |dv|."""
import numpy as np
import pytest

from gpu_common import big_case, domain_radius, gpu_config, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu

QE, ME = 1.6021766e-19, 9.109383e-31


def _check(case, parts, others=()):
    cases = [case] + [c for c, _ in others]
    ctx = G.Context([gpu_config(c, 40 + i) for i, c in enumerate(cases)], G.POTG_FP64)
    ctx.upload(0, parts.view(G.PARTICLE_DT), q=-30)
    for i, (_, p) in enumerate(others):
        ctx.upload(i + 1, p.view(G.PARTICLE_DT), q=-30)
    ctx.build_tree()
    dt = float(case["args"]["-d"])
    el = np.nonzero(parts["species"] == G.ELECTRON)[0].astype(np.uint32)
    xyz = np.stack([parts[f][el] + 0.5 * dt * parts["v" + f][el] for f in ("x", "y", "z")], 1)
    E, cnt = ctx.field_at(0, xyz, exclude=el, counts=True)
    ctx.stats_reset()
    ctx.step()
    st = ctx.stats()
    if not others:
        assert [st[k] for k in ("n_cell", "n_leaf", "n_open")] == [int(c) for c in cnt.sum(0, dtype=np.int64)]
    after, _ = ctx.download(0)
    v0 = np.stack([parts["v" + f][el] for f in ("x", "y", "z")], 1)
    v1 = np.stack([after["v" + f][el] for f in ("x", "y", "z")], 1)
    x1 = np.stack([after[f][el] for f in ("x", "y", "z")], 1)
    # reinjected electrons start anew at the boundary
    keep = np.abs(x1 - xyz - 0.5 * dt * v1).max(1) < 1e-9 * domain_radius(case)
    assert keep.mean() > 0.9
    dv = -QE / ME * dt * E
    err = np.linalg.norm(v1 - v0 - dv, axis=1)[keep]
    mag = np.linalg.norm(dv, axis=1)[keep]
    round_off = 8 * 2.0 ** -53 * (np.linalg.norm(v0, axis=1)[keep] + mag)
    assert np.all(err <= 1e-11 * np.maximum(mag, np.median(mag)) + round_off), (err / mag).max()


@pytest.mark.parametrize("N,theta,geometry,dipoles", [(500001, 0.12, 0, 0), (500002, 0.14, 1, 1),
                                                      (700001, 0.16, 0, 1)])
def test_uniform(N, theta, geometry, dipoles):
    case = dict(big_case(N, geometry=geometry, A=2.0 if geometry else 1.0, seed=21), dipoles=dipoles,
                theta=theta)
    _check(case, oracle_sim(case).particles())


def test_chain_to_a_clump():
    case = dict(big_case(500001, seed=22), dipoles=1, theta=0.15)
    parts = oracle_sim(case).particles()
    R = domain_radius(case)
    for f, c in (("x", 0.55), ("y", 1.3), ("z", 0.7)):
        parts[f][2000:] = c * R + (parts[f][2000:] - R) / 64.0
        parts["v" + f][2000:] /= 64.0
    _check(case, parts)


def test_batch_with_another_kind():
    case = dict(big_case(500001, seed=23), dipoles=0, theta=0.12)
    other = dict(big_case(20001, seed=24), theta=0.4, dipoles=1)
    _check(case, oracle_sim(case).particles(), [(other, oracle_sim(other).particles())])
