"""The work counters of point queries: n_child_visits grows with them, in every
walk's shape of a mixed context that keeps it, so that the share of lanes that
do an interaction can be read from potg_stats whatever was asked in between; a
context that starts over starts from zero."""
import numpy as np
import pytest

from gpu_common import big_case, gpu_ctx, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group,variant", [(64, 1), (64, 0)])
def test_child_visits_of_point_queries(group, variant):
    case = big_case(60001, seed=61)
    parts = oracle_sim(case).particles()
    ctx = gpu_ctx(case, parts, precision=G.POTG_MIXED)
    ctx.set_tuning(1024, group, variant)
    ctx.build_tree()
    idx = np.arange(1, 60001, 5, dtype=np.uint32)
    xyz = np.stack([parts[f][idx] for f in ("x", "y", "z")], 1)
    ctx.stats_reset()
    for rep in (1, 2):
        cnt = ctx.field_at(0, xyz, exclude=idx, counts=True)[1].sum(0, dtype=np.int64)
        st = ctx.stats()
        assert [st[k] for k in ("n_cell", "n_leaf", "n_open")] == [rep * int(c) for c in cnt]
        useful = (st["n_cell"] + st["n_leaf"]) / (64 * max(st["n_child_visits"], 1))
        assert st["n_child_visits"] > 0 and useful <= 1.0, useful
    ctx.stats_reset()
    assert ctx.stats()["n_child_visits"] == 0
