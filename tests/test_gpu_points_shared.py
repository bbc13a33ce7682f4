"""Point queries of many points at small opening angles, walked 64 a wavefront:
whether a query is (by its number of points, angle, tree and the points' order,
told apart by the ranges fetched: a range that a point opens is fetched once a
wavefront), and that fields, potentials and counts are those of each point alone
(the same points asked for a few thousand at a time), also next to points that
are no number or out of reach, and with a spheroid's analytic field.

Tolerance: both float64 walks sum the same terms, each good to a few units of
2^-53, in different orders: 1e-12 of the sum, or, where terms cancel, of the
sums' median; the float32 walks' differ by float32 roundings, 1e-5 at the median
and 1e-3 at the 99th percentile (cancelling sums)."""
import ctypes as C

import numpy as np
import pytest
import torch

from gpu_common import big_case, domain_radius, gpu_ctx, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu

PRECS = pytest.mark.parametrize("prec", [G.POTG_FP64, G.POTG_MIXED], ids=["fp64", "mixed"])


def _points(N, n, order, R, parts, seed=1):
    idx = np.random.default_rng(seed).permutation(np.arange(1, N))[:n].astype(np.uint32)
    if order == "order":
        idx = idx[np.lexsort([np.floor(parts[f][idx] / R * 20) for f in ("x", "y", "z")])]
    return idx, np.stack([parts[f][idx] for f in ("x", "y", "z")], 1)


@PRECS
@pytest.mark.parametrize("N,theta,geometry,dipoles,n,order,shared", [
    (60001, 0.0, 0, 1, 60000, "scattered", True), (60001, 0.02, 1, 1, 49152, "scattered", True),
    (200001, 0.02, 0, 0, 65536, "scattered", True), (200001, 0.06, 0, 1, 100000, "order", True),
    (200001, 0.06, 0, 1, 100000, "scattered", False), (200001, 0.02, 0, 1, 49151, "order", False),
    (200001, 0.3, 0, 1, 100000, "order", False), (20001, 0.0, 0, 1, 20000, "order", False),
    (700001, 0.2, 1, 1, 600001, "order", True)])
def test_fields_and_potentials(prec, N, theta, geometry, dipoles, n, order, shared):
    case = dict(big_case(N, geometry=geometry, A=2.0 if geometry else 1.0, seed=71), theta=theta,
                dipoles=dipoles)
    parts = oracle_sim(case).particles()
    ctx = gpu_ctx(case, parts, precision=prec, q=-30)
    ctx.build_tree()
    idx, xyz = _points(N, n, order, domain_radius(case), parts)
    ctx.stats_reset()
    E, cnt = ctx.field_at(0, xyz, exclude=idx, counts=True)
    st = ctx.stats()
    assert (4 * st["n_range_loads"] < st["n_open"]) == shared, st
    assert [st[k] for k in ("n_cell", "n_leaf", "n_open")] == [int(c) for c in cnt.sum(0, dtype=np.int64)]
    phi = ctx.phi_at(0, xyz)
    some = np.arange(0, n, max(1, n // 6000))
    E1, cnt1 = ctx.field_at(0, xyz[some], exclude=idx[some], counts=True)
    phi1 = ctx.phi_at(0, xyz[some])
    assert np.array_equal(cnt[some], cnt1)
    err, mag = np.linalg.norm(E[some] - E1, axis=1), np.linalg.norm(E1, axis=1)
    if prec == G.POTG_FP64:
        assert np.all(err <= 1e-12 * np.maximum(mag, np.median(mag)))
    else:
        assert np.median(err / mag) < 1e-5 and np.percentile(err / mag, 99) < 1e-3
    assert np.all(np.abs(phi[some] - phi1) <= 1e-12 * np.maximum(np.abs(phi1), np.median(np.abs(phi1))))


@PRECS
def test_neighbours_of_points_that_are_out_of_reach(prec):
    case = dict(big_case(60001, seed=72), theta=0.02)
    parts = oracle_sim(case).particles()
    ctx = gpu_ctx(case, parts, precision=prec, q=-30)
    ctx.build_tree()
    idx, xyz = _points(60001, 60000, "scattered", domain_radius(case), parts)
    E, cnt = ctx.field_at(0, xyz, exclude=idx, counts=True)
    phi = ctx.phi_at(0, xyz)
    bad = np.arange(17, 60000, 997)
    xyz2 = xyz.copy()
    xyz2[bad[0::2], 1] = np.nan
    xyz2[bad[1::2], 0] = 1e200
    E2, cnt2 = ctx.field_at(0, xyz2, exclude=idx, counts=True)
    phi2 = ctx.phi_at(0, xyz2)
    ok = np.setdiff1d(np.arange(60000), bad)
    assert np.array_equal(E[ok], E2[ok]) and np.array_equal(cnt[ok], cnt2[ok])
    assert np.array_equal(phi[ok], phi2[ok])
    assert np.all(np.isnan(E2[bad[0::2]])) and np.all(np.isnan(phi2[bad[0::2]]))
    assert np.array_equal(phi2[bad[1::2]], np.zeros(len(bad[1::2])))
    if prec == G.POTG_FP64:
        assert np.array_equal(E2[bad[1::2]], np.zeros((len(bad[1::2]), 3)))


@pytest.mark.parametrize("n", [65536, 49152, 40000])
def test_the_query_that_allocates_nothing_is_the_same(n):
    """Also on another stream, and captured and replayed."""
    case = dict(big_case(120001, seed=73), theta=0.015, dipoles=1)
    parts = oracle_sim(case).particles()
    ctx = gpu_ctx(case, parts, q=-30)
    ctx.build_tree()
    xyz = _points(120001, n, "order", domain_radius(case), parts)[1]
    want = ctx.phi_at(0, xyz)
    d = torch.from_numpy(xyz).cuda()
    out = torch.zeros(n, dtype=torch.float64, device="cuda")
    s = torch.cuda.Stream()

    def ask():
        stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert ctx.L.potg_phi_at_noalloc(ctx.h, 0, C.c_void_p(d.data_ptr()), n,
                                         C.c_void_p(out.data_ptr()), stream) == 0

    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        ask()
    s.synchronize()
    assert np.array_equal(out.cpu().numpy(), want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        ask()
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), want)
        assert np.array_equal(ctx.phi_at(0, xyz[:100]), ctx.phi_at(0, xyz[:100]))
    ctx.sync()
