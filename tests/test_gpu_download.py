"""Downloads return what was uploaded, in the reference's order, whatever
order the device holds it in: particle counts around a chunk of the copy (1
MB, 18724 particles), enough for two threads (16 MB), batches of unlike
instances with and without a grain in the tree, as uploaded and after a tree
build has reordered them."""
import numpy as np
import pytest

from gpu_common import big_case, gpu_config, oracle_sim

from pot_amd import potg as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [[(3, 0)], [(18724, 0)], [(18725, 1)], [(299593, 0)], [(299594, 0)],
                                   [(1200001, 0)], [(700, 0), (18725, 1), (3, 1), (40001, 0)]],
                         ids=lambda s: "-".join("%d.%d" % p for p in s))
def test_round_trip(shape):
    cases = [big_case(n, geometry=g, A=2.0 if g else 1.0, seed=n) for n, g in shape]
    parts = [oracle_sim(c).particles().view(G.PARTICLE_DT) for c in cases]
    ctx = G.Context([gpu_config(c) for c in cases], G.POTG_MIXED)
    for k, p in enumerate(parts):
        ctx.upload(k, p, q=-k - 1, m=1e-12, tot_e=k)
    for build in (False, True):
        if build:
            ctx.build_tree()
        for k, p in enumerate(parts):
            back, grain = ctx.download(k)
            assert (grain["q"], grain["tot_e"]) == (-k - 1, k)
            for f in ("x", "y", "z", "vx", "vy", "vz", "species"):
                assert np.array_equal(back[f], p[f]), (k, f, build)
