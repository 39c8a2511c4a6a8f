"""Source splits of the tiled and 16-row kernels (HOLO_FP32_SPLIT, targets too near
for the GEMM forms or off a lattice): against one split, where each result is within
the FP32-split bar of 1e-6, at the edges of the rules that choose them.
"""
import numpy as np
import pytest

from test_gpu_pairs import LAM, lattice, rel_l2, weights
from test_gpu_points import jittered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("src", [(9, 7), (64, 1), (13, 10), (64, 64), (90, 91), (130, 127)])
@pytest.mark.parametrize("M", [1, 63, 257, 4096, 4097, 140000])
def test_tile_splits(pkg, ctx, src, M):
    g = np.random.default_rng(M)
    v = (g.random((M, 3)) - 0.5) * [2e-3, 2e-3, 0] + [0, 0, 0.01]
    for u in (jittered(*src, 8e-6), lattice(*src, 8e-6, 8e-6)):
        amp, phase = weights(1, len(u))
        plan = ctx.plan(u)
        y = plan.transform(amp, phase, v, 1, LAM, pkg.FP32_SPLIT)
        pkg.set_option("splits", 1)
        one = plan.transform(amp, phase, v, 1, LAM, pkg.FP32_SPLIT)
        pkg.set_option("splits", 0)
        assert rel_l2(y, one) <= 1e-6
