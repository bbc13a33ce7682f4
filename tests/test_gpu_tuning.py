"""Launch parameters are what runs and what is reported: a float64 context whose
wavefronts share tiles has 8 blocks per CU by default, which are launched as
they are reported and as they are set; and potg_tune keeps the settings that
have no effect on a context (the grid of a walk of 2 targets a wavefront, the
radix sort's tile where keys are merged) instead of picking among equal
launches by their timing noise."""
import pytest
import torch

from gpu_common import big_case, gpu_config, gpu_ctx, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu


def _cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


def test_default_grid_of_shared_tiles():
    for N, theta, bpc in ((500001, 0.12, 8), (200001, 0.02, 8), (500001, 0.5, 4)):
        ctx = G.Context([gpu_config(dict(big_case(N), theta=theta))], G.POTG_FP64)
        assert ctx.tuning()["walk_blocks"] == bpc * _cus(), (N, theta)
        ctx.close()


@pytest.mark.parametrize("prec", [G.POTG_FP64, G.POTG_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("tile", [2048, 4096])
def test_tune_keeps_what_has_no_effect(prec, tile):
    case = big_case(60001, seed=23)
    ctx = gpu_ctx(case, oracle_sim(case).particles(), precision=prec, seed=3)
    ctx.set_tuning(1000, 64, 0, tile)
    t = ctx.tune()
    assert t["sort_tile"] == tile and t["walk_ms"] > 0
    if prec == G.POTG_FP64:
        assert t["walk_blocks"] == 1000 == ctx.tuning()["walk_blocks"]


def test_tune_chooses_the_grid_of_shared_tiles():
    case = dict(big_case(200001, seed=24), theta=0.04)
    ctx = gpu_ctx(case, oracle_sim(case).particles(), seed=3)
    ctx.set_tuning(100, 64, 0)
    assert ctx.tune()["walk_blocks"] in [b * _cus() for b in (2, 4, 8, 16)]
