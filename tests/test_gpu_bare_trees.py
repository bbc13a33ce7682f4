"""Trees without internal nodes, an empty cell or one leaf for a root: a
spheroid grain alone (it is no part of the tree) or with one particle, and a
spherical grain alone, first, between and behind larger instances and with
nothing else in the context.  Their potentials and fields are one point's, and
every instance of the batch has the tree, fields, potentials and steps (chi_b
and energies among them) of the same one alone, bit for bit."""
import numpy as np
import pytest

from gpu_common import big_case, domain_radius, gpu_config, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu

K = 1.6021766e-19 / (4.0 * np.pi * 8.85419e-12)
GEN = big_case(3001, seed=51)
R = domain_radius(GEN)


def _bare(N, geometry, dipoles, integrator):
    """a case of N particles in GEN's domain: the grain and N - 1 ions"""
    case = dict(GEN, geometry=geometry, dipoles=dipoles, integrator=integrator,
                args=dict(GEN["args"], **{"-N": str(N)}, **({"-A": "2.0"} if geometry else {})))
    parts = np.zeros(N, G.PARTICLE_DT)
    for f in ("x", "y", "z"):
        parts[f] = R
    parts["x"][1:] = 1.4 * R
    parts["vy"][1:] = 1e3
    parts["species"][1:] = G.ION
    return case, parts


def _large(N, geometry, dipoles, integrator):
    case = dict(big_case(N, geometry=geometry, A=2.0 if geometry else 1.0, seed=N), dipoles=dipoles,
                integrator=integrator)
    return case, oracle_sim(case).particles().view(G.PARTICLE_DT)


def _ctx(insts, prec, seeds, q):
    ctx = G.Context([gpu_config(c, s) for (c, _), s in zip(insts, seeds)], prec)
    for k, (_, p) in enumerate(insts):
        ctx.upload(k, p, q=q, t=18, chi_b=-0.5)
    # so few particles' chi_b may bar a species: such an instance retires
    ctx.set_retire(True)
    return ctx


def _queries(ctx, k, case, n):
    rad = domain_radius(case)
    pts = rad + 0.8 * rad * np.random.default_rng(3).uniform(-1.0, 1.0, (9, 3))
    out = [ctx.phi_at(k, pts)]
    out += ctx.field_at(k, pts, counts=True)
    out += ctx.field_at(k, pts, exclude=np.arange(9, dtype=np.uint32) % n, counts=True)
    t = ctx.tree_canon(k)
    out += [t[f] for f in ("depth", "is_leaf", "q", "aq", "nchild", "c", "size2")]
    out += [t["part"][t["is_leaf"] == 1], ctx.tree_dipoles(k)]
    return out


@pytest.mark.parametrize("prec", [G.POTG_FP64, G.POTG_MIXED, G.POTG_MIXED_GROUP],
                         ids=["fp64", "mixed", "mixed_group"])
@pytest.mark.parametrize("dipoles", [0, 1], ids=["monopole", "dipoles"])
@pytest.mark.parametrize("integrator", [G.POTG_BORIS, G.POTG_VERLET], ids=["boris", "verlet"])
@pytest.mark.parametrize("larger", [True, False], ids=["among_larger", "only"])
def test_batch_of_bare_trees_is_each_alone(prec, dipoles, integrator, larger):
    rest = (dipoles, integrator)
    insts = [_bare(1, 1, *rest), _bare(2, 1, *rest), _bare(1, 0, *rest)]
    if larger:
        insts = [insts[0], _large(3001, 0, *rest), insts[1], insts[2], _large(701, 1, *rest),
                 _bare(1, 1, *rest)]
    seeds = range(60, 60 + len(insts))
    batch = _ctx(insts, prec, seeds, -7)
    ones = [_ctx([i], prec, [s], -7) for i, s in zip(insts, seeds)]
    for c in [batch] + ones:
        c.build_tree()
    for k, (case, p) in enumerate(insts):
        for a, b in zip(_queries(batch, k, case, len(p)), _queries(ones[k], 0, case, len(p))):
            assert np.array_equal(a, b) and np.all(np.isfinite(a)), k
    for epe in (0, 1, 0):  # steps 19, 20 (chi_b is taken) and 21
        out = batch.step(epe)
        for k, one in enumerate(ones):
            assert one.step(epe)[0] == out[k], k
    for k, one in enumerate(ones):
        (pb, gb), (po, go) = batch.download(k), one.download(0)
        assert np.array_equal(pb.view(np.uint8), po.view(np.uint8)) and gb == go, k
        assert batch.retired(k) == one.retired(0), k
    for c in [batch] + ones:  # the same captured
        c.run(2)
    for k, one in enumerate(ones):
        assert np.array_equal(batch.download(k)[0], one.download(0)[0]), k


@pytest.mark.parametrize("prec", [G.POTG_FP64, G.POTG_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("N,geometry,q", [(1, 0, -7), (2, 1, 0), (1, 1, 0)])
def test_one_point_and_none(prec, N, geometry, q):
    """Tolerance: one term, some roundings of its precision (the float32 walk's
    coordinates, in units of R, are good to 6e-8 each)."""
    case, parts = _bare(N, geometry, 1, G.POTG_BORIS)
    ctx = _ctx([(case, parts)], prec, [1], q)
    ctx.build_tree()
    pts = R + 0.8 * R * np.random.default_rng(4).uniform(-1.0, 1.0, (33, 3))
    src, ch = ((R, R, R), float(q)) if geometry == 0 else ((1.4 * R, R, R), float(N - 1))
    d = pts - np.array(src)
    r = np.sqrt((d * d).sum(1) + float(case["args"]["-s"]) ** 2)
    phi, E = ctx.phi_at(0, pts), ctx.field_at(0, pts)
    want = K * ch * d / r[:, None] ** 3
    tol = 1e-14 if prec == G.POTG_FP64 else 1e-6 * R / r[:, None]
    assert np.all(np.abs(phi - K * ch / r) <= 1e-14 * np.abs(K * ch / r))
    assert np.all(np.abs(E - want) <= tol * np.linalg.norm(want, axis=1)[:, None])
