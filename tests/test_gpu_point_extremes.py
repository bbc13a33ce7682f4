"""Point queries where float32 or float64 arithmetic runs out: points on top of
particles under a softening whose cube has no float32 reciprocal; points (and
half-drifted particles) so far out that their squared distance overflows, for
which every term is zero; a softening whose square overflows; and points that
are no number.  Every cell opens for those and every leaf is met, as in the
reference's opening test, which no comparison with a NaN passes."""
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


@pytest.mark.parametrize("prec", [G.POTG_FP64, G.POTG_MIXED], ids=["fp64", "mixed"])
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


@pytest.mark.parametrize("theta", [0.0, 0.5])
@pytest.mark.parametrize("dipoles", [0, 1], ids=["monopole", "dipoles"])
def test_squared_distances_that_overflow(theta, dipoles):
    case = dict(big_case(3001, seed=15), theta=theta, dipoles=dipoles)
    parts = oracle_sim(case).particles()
    ctx = gpu_ctx(case, parts, q=-9)
    ctx.build_tree()
    pts = np.array([[1e155, 1.0, -2.0], [0.0, -1e200, 3.0], [1e300, 1e300, 1e300], [1.0, 1.0, 1e154]])
    E, c = ctx.field_at(0, pts, counts=True)
    assert np.array_equal(E[:3], np.zeros((3, 3))) and np.all(np.abs(E[3]) < 1e-300)
    assert np.array_equal(ctx.phi_at(0, pts[:3]), np.zeros(3))
    if theta == 0.0:  # zero times an infinite distance accepts no cell
        assert np.all(c[:3, 1] == 3001) and np.all(c[:3, 0] == 0)
    if not dipoles:
        far = ctx.phi_at(0, [[np.inf, 0.0, 0.0], [0.0, -np.inf, np.inf]])
        assert np.array_equal(far, np.zeros(2))


def test_softening_whose_square_overflows():
    case = big_case(3001, seed=16)
    case["args"]["-s"] = "1e160"
    parts = oracle_sim(case).particles()
    idx = np.arange(1, 3001, 11, dtype=np.uint32)
    xyz = np.stack([parts[f][idx] for f in ("x", "y", "z")], 1)
    E = gpu_ctx(case, parts, q=-9).direct_sum(0, idx)
    assert np.array_equal(E, np.zeros_like(E))
    # the cells are not softened: those alone are left
    case["theta"] = 0.0
    ctx = gpu_ctx(case, parts, q=-9)
    ctx.build_tree()
    assert np.array_equal(ctx.field_at(0, xyz, exclude=idx), np.zeros_like(E))
    assert np.array_equal(ctx.phi_at(0, xyz), np.zeros(len(idx)))
    case["theta"] = 0.5
    ctx = gpu_ctx(case, parts, q=-9)
    ctx.build_tree()
    E = ctx.field_at(0, xyz, exclude=idx)
    assert np.all(np.isfinite(E)) and np.all(np.isfinite(ctx.phi_at(0, xyz)))


@pytest.mark.parametrize("N,theta", [(4001, 0.5), (500001, 0.12)], ids=["few", "shared"])
def test_a_particle_that_leaves_at_any_speed(N, theta):
    """Electrons so fast that the squared distances of their half-drifted
    positions overflow feel no field and come in again at the boundary."""
    case = dict(big_case(N, seed=17), theta=theta)
    parts = oracle_sim(case).particles()
    el = np.nonzero(parts["species"] == G.ELECTRON)[0]
    for k, f in enumerate(("vx", "vy", "vz")):
        parts[f][el[100 + k]] = (-1.0) ** k * 1e180
    ctx = gpu_ctx(case, parts, q=-9)
    ctx.step()
    ctx.step(1)
    p, g = ctx.download(0)
    assert all(np.all(np.isfinite(p[f])) for f in ("x", "y", "z", "vx", "vy", "vz"))
    assert np.all(np.isfinite(g["epe"])) and np.all(np.abs(p["vx"]) < 1e100)
