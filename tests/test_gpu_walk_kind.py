"""Which float64 walk an instance takes: 2 targets a wavefront, or, where the
opening angle is small for the size, 64 targets shared by four wavefronts.  The
counters tell the two apart: a range that a target opens is fetched once for
the targets of a wavefront, so 2 targets fetch at least half as many ranges as
targets open, and 64 a small part of that, although the walks' sets are the
same.  At theta = 0 every target meets every particle, and a walk of 2 targets
takes several times one of 64 from some 100000 particles on.  Where the walks
are new to a size, the step's field is the point field (as in
test_gpu_walk_split.py); and the energies of a record step, whose walk has 1 or
64 targets a wavefront, are those of the potentials at the particles.  From 2M
particles on a tile of 64 has one wavefront.  The shared tiles' partial sums are
held for 2^21 targets at a time, so that batches of any size find the memory."""
import numpy as np
import pytest
import torch

from gpu_common import big_case, gpu_config, gpu_ctx, oracle_sim
from test_gpu_walk_split import _check

from pot_amd import potg as G

pytestmark = pytest.mark.gpu


def shares_tiles(ctx):
    """of a context with one float64 instance, after steps since its counters
    were reset"""
    st = ctx.stats()
    return 4 * st["n_range_loads"] < st["n_open"]


@pytest.mark.parametrize("N,theta,dipoles,shared", [
    (20001, 0.0, 1, False), (120001, 0.0, 1, True), (200001, 0.03, 0, True),
    (200001, 0.05, 1, True), (200001, 0.12, 1, False), (300001, 0.0, 0, True),
    (450001, 0.05, 1, True), (450001, 0.11, 0, True), (450001, 0.2, 1, False),
    (500001, 0.12, 0, True), (500001, 0.14, 1, True), (500001, 0.2, 1, False)])
def test_kind_by_angle_and_size(N, theta, dipoles, shared):
    case = dict(big_case(N, seed=31), theta=theta, dipoles=dipoles)
    ctx = gpu_ctx(case, oracle_sim(case).particles(), q=-30)
    ctx.step()
    assert shares_tiles(ctx) == shared, ctx.stats()


@pytest.mark.parametrize("N,theta,geometry,dipoles", [(120002, 0.02, 0, 1), (200001, 0.0, 0, 0),
                                                      (300001, 0.08, 1, 1)])
def test_shared_tiles_of_smaller_instances(N, theta, geometry, dipoles):
    case = dict(big_case(N, geometry=geometry, A=2.0 if geometry else 1.0, seed=32), theta=theta,
                dipoles=dipoles)
    _check(case, oracle_sim(case).particles())


QE, K4PE0 = 1.6021766e-19, 4.0 * np.pi * 8.85419e-12


@pytest.mark.parametrize("prec", [G.POTG_FP64, G.POTG_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("N,theta,dipoles", [(60001, 0.01, 1), (60001, 0.2, 1), (250001, 0.09, 0),
                                             (500001, 0.12, 1), (500001, 0.13, 0)])
def test_energies_are_the_potentials(prec, N, theta, dipoles):
    """Particles at rest are not drifted, so a particle's potential is that of a
    point query at its place but for its own leaf's q / soft.  (At these angles
    no cell that holds a target is far enough from it to be taken whole.)  Both
    walks are exact to some roundings of each term: 1e-13 of the terms' sum,
    which is below that of the leaves' own plus N / R each."""
    case = dict(big_case(N, seed=33), theta=theta, dipoles=dipoles)
    parts = oracle_sim(case).particles()
    for f in ("vx", "vy", "vz"):
        parts[f] = 0.0
    ctx = gpu_ctx(case, parts, precision=prec, q=-30)
    ctx.build_tree()
    phi = ctx.phi_at(0, np.stack([parts[f] for f in ("x", "y", "z")], 1))
    ctx = gpu_ctx(case, parts, precision=prec, q=-30)
    ctx.step(1)
    epe = ctx.download(0)[1]["epe"]
    q = np.array([-30.0, 1.0, -1.0])[parts["species"]]
    own = QE * q / (K4PE0 * float(case["args"]["-s"]))
    R = float(case["args"]["-r"]) * float(case["args"]["-m"])
    for s in (G.ION, G.ELECTRON):
        k = parts["species"] == s
        want = float((QE * q[k] * (phi[k] - own[k])).sum())
        mag = float((QE * (np.abs(own[k]) + QE / K4PE0 * 4.0 * N / R)).sum())
        assert abs(epe[s] - want) <= 1e-13 * mag, (s, epe[s], want, mag)


@pytest.mark.parametrize("N,theta", [(2000001, 0.2), (2100001, 0.24)])
def test_whole_tiles_of_large_instances(N, theta):
    case = dict(big_case(N, seed=34), theta=theta, dipoles=1)
    _check(case, oracle_sim(case).particles())


def _bytes_of(configs):
    free0 = torch.cuda.mem_get_info()[0]
    ctx = G.Context(configs, G.POTG_FP64)
    used = free0 - torch.cuda.mem_get_info()[0]
    ctx.close()
    return used


def test_memory_of_shared_tiles_is_bounded():
    """30M particles in instances that share tiles, against the same with a
    wide angle: 96 bytes for each of 2^21 targets and allocation granules more."""
    cases = [dict(big_case(1000001, seed=35), theta=t) for t in (0.1, 0.9)]
    shared, few = (_bytes_of([gpu_config(c)] * 30) for c in cases)
    assert 0 <= shared - few <= 96 * 2 ** 21 + 2 ** 25, (shared, few)


def test_batch_of_more_targets_than_parts():
    """Five instances whose targets, stepped all at once (step 42, when the ions
    are due), fill the parts two and a half times, one of them walked 2 by 2:
    each ends as it does alone, bit for bit."""
    case = dict(big_case(1000001, seed=36), theta=0.15)
    wide = dict(big_case(300001, seed=37), theta=0.9)
    parts, pw = oracle_sim(case).particles(), oracle_sim(wide).particles()
    batch = G.Context([gpu_config(case, 7)] * 3 + [gpu_config(wide, 8)] + [gpu_config(case, 7)] * 2,
                      G.POTG_FP64)
    one = [G.Context([gpu_config(c, s)], G.POTG_FP64) for c, s in ((case, 7), (wide, 8))]
    for k in (0, 1, 2, 4, 5):
        batch.upload(k, parts.view(G.PARTICLE_DT), q=-30, t=41)
    batch.upload(3, pw.view(G.PARTICLE_DT), q=-30, t=41)
    one[0].upload(0, parts.view(G.PARTICLE_DT), q=-30, t=41)
    one[1].upload(0, pw.view(G.PARTICLE_DT), q=-30, t=41)
    out = batch.step()
    assert sum(o["n_pushed"] for o in out) > 2.5 * 2 ** 21
    want = []
    for c in one:
        c.step()
        want.append(c.download(0))
    for k in range(6):
        p, g = batch.download(k)
        pw_, gw = want[k == 3]
        assert np.array_equal(p.view(np.uint8), pw_.view(np.uint8)) and g == gw, k


def test_all_kinds_in_one_context():
    """A tile for each wavefront, shared tiles and 2 targets a wavefront in one
    context, whose instances start anywhere in a tile: two steps, the second with
    its energies (1 or 64 targets a wavefront), end as each does alone, bit for
    bit."""
    cases = [dict(big_case(3002, seed=42), theta=0.7), dict(big_case(2000011, seed=43), theta=0.22),
             dict(big_case(500001, seed=44), theta=0.13, dipoles=1),
             dict(big_case(20001, seed=45), theta=0.4, dipoles=1),
             dict(big_case(150001, geometry=1, A=2.0, seed=46), theta=0.04, dipoles=1)]
    states = [oracle_sim(c).particles().view(G.PARTICLE_DT) for c in cases]
    batch = G.Context([gpu_config(c, 50 + i) for i, c in enumerate(cases)], G.POTG_FP64)
    ones = [G.Context([gpu_config(c, 50 + i)], G.POTG_FP64) for i, c in enumerate(cases)]
    for i, p in enumerate(states):
        batch.upload(i, p, q=-30)
        ones[i].upload(0, p, q=-30)
    for epe in (0, 1):
        out = batch.step(epe)
        for i, one in enumerate(ones):
            assert one.step(epe)[0] == out[i], i
    for i, one in enumerate(ones):
        (pb, gb), (po, go) = batch.download(i), one.download(0)
        assert np.array_equal(pb.view(np.uint8), po.view(np.uint8)) and gb == go, i


@pytest.mark.parametrize("n_el", [1, 2, 3, 5, 63, 64, 65, 130, 131])
@pytest.mark.parametrize("dipoles", [0, 1], ids=["monopole", "dipoles"])
def test_pairs_of_targets(n_el, dipoles):
    """Any number of targets, the last of an odd number alone with a wavefront:
    electrons at rest are moved by dt times the point field (a few roundings,
    and the sums' order)."""
    case = dict(big_case(3001, seed=47), dipoles=dipoles)
    case["args"]["-N"] = str(n_el + 1)
    R = float(case["args"]["-r"]) * float(case["args"]["-m"])
    parts = np.zeros(n_el + 1, G.PARTICLE_DT)
    rng = np.random.default_rng(n_el)
    for f in ("x", "y", "z"):
        parts[f] = R
        parts[f][1:] = R + 0.5 * R * rng.uniform(-1.0, 1.0, n_el)
    parts["species"][1:] = G.ELECTRON
    ctx = gpu_ctx(case, parts, q=9)
    ctx.build_tree()
    el = np.arange(1, n_el + 1, dtype=np.uint32)
    E, cnt = ctx.field_at(0, np.stack([parts[f][1:] for f in ("x", "y", "z")], 1), exclude=el, counts=True)
    ctx.stats_reset()
    ctx.step()
    st = ctx.stats()
    assert [st[k] for k in ("n_cell", "n_leaf", "n_open")] == [int(c) for c in cnt.sum(0, dtype=np.int64)]
    p = ctx.download(0)[0]
    v = np.stack([p["v" + f][1:] for f in ("x", "y", "z")], 1)
    dv = -QE / 9.109383e-31 * float(case["args"]["-d"]) * E
    assert np.all(np.linalg.norm(v - dv, axis=1) <= 1e-11 * np.linalg.norm(dv, axis=1))
