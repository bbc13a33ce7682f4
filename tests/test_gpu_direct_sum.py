"""potg_direct_sum at the edges of its split over the sources: particle counts
at and around the 256-particle chunks, from one target to more than a block
of them, every grain shape's source list, an uncharged grain and no
softening, against the same sum in numpy float64.

Tolerance: a term is off by at most 8 units of 2^-53 of itself (the refined
reciprocal square root, the products), numpy's by less, and a float64 sum of
N terms in any order by at most N units of the sum of their magnitudes."""
import numpy as np
import pytest

from gpu_common import big_case, gpu_config, gpu_ctx, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu

QE, EPS0 = 1.6021766e-19, 8.85419e-12


def _numpy_sum(parts, cfg, idx, q):
    x = np.stack([parts["x"], parts["y"], parts["z"]], 1)
    ch = np.array([float(q), 1.0, -1.0])[parts["species"]]
    if cfg.geometry != G.POTG_SPHERE:
        ch[0] = 0.0  # the spheroid grain is no point source
    E, mag = np.zeros((len(idx), 3)), np.zeros(len(idx))
    for k, i in enumerate(idx):
        d = x[i] - x
        r2 = (d * d).sum(1) + cfg.soft ** 2
        use = (np.arange(len(x)) != i) & (ch != 0.0)
        w = ch[use] / (r2[use] * np.sqrt(r2[use]))
        E[k] = (w[:, None] * d[use]).sum(0)
        mag[k] = np.linalg.norm(w[:, None] * d[use], axis=1).sum()
    K = QE / (4.0 * np.pi * EPS0)
    return K * E, K * mag


@pytest.mark.parametrize("N,n,q,soft", [(3, 1, -5, None), (256, 3, -5, None), (257, 256, 0, None),
                                        (258, 257, -5, 0.0), (513, 1, 0, 0.0), (4099, 700, -70, None),
                                        (20001, 64, 3, None)])
def test_direct_sum_at_chunk_edges(N, n, q, soft):
    case = big_case(N, seed=7)
    if soft is not None:
        case["args"]["-s"] = repr(soft)
    parts = oracle_sim(case).particles()
    ctx = gpu_ctx(case, parts, q=q)
    if N > 1000:
        ctx.build_tree()  # sorted state: the sources come through the inverse
    idx = np.random.default_rng(N).integers(1, N, size=n).astype(np.uint32)
    idx[-1] = N - 1
    E = ctx.direct_sum(0, idx)
    want, mag = _numpy_sum(parts, gpu_config(case), idx, q)
    err = np.abs(E - want).max(1)
    assert np.all(err <= (16 + 2 * N) * 2.0 ** -53 * mag), (err / mag).max()


@pytest.mark.parametrize("geometry,A", [(1, 2.0), (2, 0.5)], ids=["prolate", "oblate"])
def test_direct_sum_spheroid_has_no_grain_source(geometry, A):
    """With an uncharged spheroid the analytic term is zero: the sum over the
    other particles alone."""
    case = big_case(769, geometry=geometry, A=A, seed=8)
    parts = oracle_sim(case).particles()
    ctx = gpu_ctx(case, parts, q=0)
    idx = np.arange(1, 769, dtype=np.uint32)
    E = ctx.direct_sum(0, idx)
    want, mag = _numpy_sum(parts, gpu_config(case), idx, 0)
    err = np.abs(E - want).max(1)
    assert np.all(err <= (16 + 2 * 769) * 2.0 ** -53 * mag), (err / mag).max()
