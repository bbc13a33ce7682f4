"""The walks that share a wavefront between 64 targets, at a size and opening
angle that select them (small theta, hundreds of thousands of particles):
the velocities a step gives its electrons against the field that point
queries -- the walk of one target per wavefront, itself checked against the
oracle -- return at the same half-drifted positions, with the same interaction
counts; and a context holding an instance of either kind against each alone.

Tolerance: without a magnetic field a step turns v into v + dt q E / m exactly
but for a few roundings of float64 (2^-53 of |v| + |dv| each), and the two
walks sum the same terms in different orders: 1e-11 of |dv| for the float64
walk; the float32 walk differs by float32 roundings, 1e-5 of |dv| for the
median and 1e-3 at the 99th percentile (cancelling sums)."""
import numpy as np
import pytest

from gpu_common import big_case, domain_radius, gpu_config, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu

QE, ME = 1.6021766e-19, 9.109383e-31


def _ctx(cases, states, prec):
    ctx = G.Context([gpu_config(c, 40 + i) for i, c in enumerate(cases)], prec)
    for i, p in enumerate(states):
        ctx.upload(i, p.view(G.PARTICLE_DT), q=-30)
    return ctx


@pytest.mark.parametrize("prec", [G.POTG_FP64, G.POTG_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("geometry,A,dipoles", [(0, 1.0, 1), (0, 1.0, 0), (1, 2.0, 1)],
                         ids=["dipoles", "monopole", "prolate_dipoles"])
def test_step_field_is_the_point_field(prec, geometry, A, dipoles):
    case = dict(big_case(260003, geometry=geometry, A=A, seed=21), dipoles=dipoles, theta=0.16)
    parts = oracle_sim(case).particles()
    ctx = _ctx([case], [parts], prec)
    ctx.build_tree()
    dt = float(case["args"]["-d"])
    el = np.nonzero(parts["species"] == G.ELECTRON)[0].astype(np.uint32)
    xyz = np.stack([parts[f][el] + 0.5 * dt * parts["v" + f][el] for f in ("x", "y", "z")], 1)
    ctx.stats_reset()
    E, cnt = ctx.field_at(0, xyz, exclude=el, counts=True)
    ctx.stats_reset()
    ctx.step()
    st = ctx.stats()
    after, _ = ctx.download(0)
    v0 = np.stack([parts["v" + f][el] for f in ("x", "y", "z")], 1)
    v1 = np.stack([after["v" + f][el] for f in ("x", "y", "z")], 1)
    dv = -QE / ME * dt * E
    # reinjected electrons start anew at the boundary
    x1 = np.stack([after[f][el] for f in ("x", "y", "z")], 1)
    keep = np.abs(x1 - xyz).max(1) < 0.02 * domain_radius(case)
    assert keep.mean() > 0.95
    err = np.linalg.norm(v1 - v0 - dv, axis=1)[keep]
    mag = np.linalg.norm(dv, axis=1)[keep]
    if prec == G.POTG_FP64:
        assert [st[k] for k in ("n_cell", "n_leaf", "n_open")] == [int(c) for c in cnt.sum(0, dtype=np.int64)]
        round_off = 8 * 2.0 ** -53 * (np.linalg.norm(v0, axis=1)[keep] + mag)
        assert np.all(err <= 1e-11 * mag + round_off), (err / mag).max()
    else:
        # the float32 sums differ in order only: the counts are the same
        assert [st[k] for k in ("n_cell", "n_leaf", "n_open")] == [int(c) for c in cnt.sum(0, dtype=np.int64)]
        assert np.median(err / mag) < 1e-5 and np.percentile(err / mag, 99) < 1e-3


@pytest.mark.parametrize("prec", [G.POTG_FP64, G.POTG_MIXED], ids=["fp64", "mixed"])
def test_both_kinds_in_one_context(prec):
    """A large instance with a small opening angle, a small one and one with a
    large opening angle: two steps (with potential energies) of the batch and
    of each alone end in the same states bit for bit."""
    cases = [dict(big_case(3001, seed=22), theta=0.7), dict(big_case(260003, seed=23), theta=0.15),
             dict(big_case(20001, seed=24), theta=0.4, dipoles=1)]
    states = [oracle_sim(c).particles() for c in cases]
    batch = _ctx(cases, states, prec)
    batch.set_tuning(1024, 64, 1 if prec == G.POTG_MIXED else 0)
    singles = []
    for i, c in enumerate(cases):
        s = G.Context([gpu_config(c, 40 + i)], prec)
        s.upload(0, states[i].view(G.PARTICLE_DT), q=-30)
        s.set_tuning(1024, 64, 1 if prec == G.POTG_MIXED else 0)
        singles.append(s)
    for epe in (0, 1):
        batch.step(epe)
        for s in singles:
            s.step(epe)
    for i, s in enumerate(singles):
        pb, gb = batch.download(i)
        ps, gs = s.download(0)
        assert np.array_equal(pb.view(np.uint8), ps.view(np.uint8)), i
        assert gb == gs, i
