"""Monte Carlo draws split over workgroups where few targets leave the chip idle:
the indices and the sum of a target's draws stay those of the FP64 oracle (1e-12,
FP32-split 1e-6), at the edges of a split's draws and of the targets' workgroups.
"""
import numpy as np
import pytest

from test_gpu_mc_lattice import LAM, product_grid, rel_l2, targets, weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 63, 64, 127, 129, 255, 256, 257, 1031])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("M, passes", [(1, 0), (257, 3), (1025, 0)])
def test_mc_splits(pkg, ctx, oracle, K, shared, M, passes):
    u = product_grid(np.arange(37) * 8e-6, np.arange(29) * 9e-6, 0.0)
    amp, phase = weights(1, len(u))
    v = targets(2, M)
    pkg.set_option("mc_passes", passes)
    y64 = ctx.transform_mc(amp, phase, u, v, K, 11, -1, LAM, pkg.FP64, shared=shared)
    y32 = ctx.transform_mc(amp, phase, u, v, K, 11, -1, LAM, pkg.FP32_SPLIT, shared=shared)
    pkg.set_option("mc_passes", 0)
    sub = np.unique(np.concatenate([[0, M - 1], np.arange(0, M, 97)]))
    ref = oracle.transform_mc(-1, LAM, amp, phase, u, v, K, 11, targets=sub, shared=shared)
    assert rel_l2(y64[sub], ref) <= 1e-12
    assert rel_l2(y32[sub], ref) <= 1e-6
