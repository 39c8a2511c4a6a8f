"""Options that set how a call is split take effect at every size: another count sums
in another order, so the bits differ, and each result stays within its bar (FP32-split
1e-6, FP64 1e-12) of the FP64 oracle.  FP64 sums of FP32 values are mostly exact, in
any order, so the FP32-split far form shows a split only where its two-tile FP32 runs
move: here splits of three tiles.
"""
import numpy as np
import pytest

from test_gpu_pairs import LAM, lattice, rel_l2, weights
from test_gpu_points import jittered

pytestmark = pytest.mark.gpu


def scattered(M, z):
    g = np.random.default_rng(M)
    return (g.random((M, 3)) - 0.5) * [2e-3, 2e-3, 0] + [0, 0, z]


SOURCES = {
    "18 tiles": lambda: lattice(40, 72, 8e-6, 8e-6),
    "24 tiles and a tail": lambda: np.concatenate(
        [lattice(64, 96, 8e-6, 8e-6), scattered(40, 0.0)]),
    "padded, a tail": lambda: np.concatenate([lattice(50, 70, 8e-6, 8e-6), scattered(40, 0.0)]),
    "jittered": lambda: jittered(40, 36, 8e-6),
}


# the far form and exact pairs of the 16-row and tiled kernels; automatic splits too
@pytest.mark.parametrize("case", SOURCES)
@pytest.mark.parametrize("z", [0.3, 0.01])
@pytest.mark.parametrize("M", [257, 4097])
def test_splits(pkg, ctx, oracle, case, z, M):
    u, v = SOURCES[case](), scattered(M, z)
    amp, phase = weights(1, len(u))
    plan = ctx.plan(u)
    sub = np.arange(0, M, 13)
    ref = oracle.transform_full(1, LAM, amp, phase, u, v[sub])
    y = {}
    for splits in (1, 3, 4, 0):
        pkg.set_option("splits", splits)
        y[splits] = plan.transform(amp, phase, v, 1, LAM, pkg.FP32_SPLIT)
        assert rel_l2(y[splits][sub], ref) <= 1e-6
    if z == 0.3:
        assert not np.array_equal(y[1], y[3 if case == "18 tiles" else 4])


# FP64: fewer ranges by default where one round of workgroups holds the call (M = 300)
@pytest.mark.parametrize("M", [300, 70000])
def test_mc_passes_fp64(pkg, ctx, oracle, M):
    u, v, K = lattice(64, 60, 8e-6, 8e-6), scattered(M, 0.3), 200
    amp, phase = weights(2, len(u))
    sub = np.arange(0, M, max(1, M // 200))
    ref = oracle.transform_mc(1, LAM, amp, phase, u, v, K, 5, targets=sub)
    y = {}
    for passes in (3, 8, 13, 64):
        pkg.set_option("mc_passes", passes)
        y[passes] = ctx.transform_mc(amp, phase, u, v, K, 5, 1, LAM, pkg.FP64)
        assert rel_l2(y[passes][sub], ref) <= 1e-12
    for a, b in ((3, 8), (8, 13), (13, 64)):
        assert not np.array_equal(y[a], y[b])
