"""Point queries where float32 or float64 arithmetic runs out: points on top of
particles under a softening whose cube has no float32 reciprocal, and points
that are no number.  Every cell opens for those and every leaf is met, as in
the reference's opening test, which no comparison with a NaN passes."""
import numpy as np
import pytest

from gpu_common import big_case, domain_radius, gpu_ctx, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("soft_over_R", [0.0, 1e-15, 1e-12, 1e-4])
@pytest.mark.parametrize("dipoles", [0, 1], ids=["monopole", "dipoles"])
def test_a_particle_under_the_point_adds_nothing(soft_over_R, dipoles):
    """The float32 field at particles that are not excluded is the one with
    the particle excluded, bit for bit, the counts too."""
    case = dict(big_case(4001, seed=13), dipoles=dipoles)
    case["args"]["-s"] = repr(soft_over_R * domain_radius(case))
    parts = oracle_sim(case).particles()
    idx = np.arange(1, 4001, 7, dtype=np.uint32)
    xyz = np.stack([parts[f][idx] for f in ("x", "y", "z")], 1)
    ctx = gpu_ctx(case, parts, precision=G.POTG_MIXED, q=-9)
    ctx.build_tree()
    E0, c0 = ctx.field_at(0, xyz, exclude=idx, counts=True)
    E1, c1 = ctx.field_at(0, xyz, counts=True)
    assert np.all(np.isfinite(E0))
    assert np.array_equal(E0, E1) and np.array_equal(c0, c1)


@pytest.mark.parametrize("prec", [G.POTG_MIXED], ids=["mixed"])
def test_a_point_that_is_no_number(prec):
    case = big_case(3001, seed=14)
    parts = oracle_sim(case).particles()
    ctx = gpu_ctx(case, parts, precision=prec, q=-9)
    ctx.build_tree()
    R = domain_radius(case)
    E, c = ctx.field_at(0, [[R, np.nan, R]], counts=True)
    n_int = int((ctx.tree_canon(0)["is_leaf"] == 0).sum())
    assert np.all(np.isnan(E))
    assert c.tolist() == [[0, 3001, n_int]]
