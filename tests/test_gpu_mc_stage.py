"""Per-target FP32-split Monte Carlo past the draw counts from which product grids
take the kernel that stages their row and column tables in LDS and other sources
the general one: both against the FP64 estimator of the same indices (1e-6), and
bit for bit whether positions come from the tables or the records (option
"mc_lattice").
"""
import numpy as np
import pytest

from test_gpu_mc_lattice import LAM, both, product_grid, rel_l2, targets, weights

pytestmark = pytest.mark.gpu


def plane(nx, ny, p=8e-6):
    return product_grid((np.arange(nx) - nx / 2) * p, (np.arange(ny) - ny / 2) * p, 0.0)


def jittered(nx, ny):
    u = plane(nx, ny)
    u[:, :2] += (np.random.default_rng(3).random((len(u), 2)) - 0.5) * 7e-6
    return u


CASES = {
    "staged, two ranges": lambda w: plane(760, 700),
    "staged, one range": lambda w: plane(640, 625),
    "the widest table": lambda w: plane(170, 2386),
    "too wide": lambda w: plane(160, 2558),
    "one column": lambda w: plane(400001, 1),
    "padded": lambda w: w.reference_plane(480007, 10e-3, 0.0, 1.3),
    "jittered": lambda w: jittered(700, 660),
}


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("M, K", [(4133, 1031), (200100, 170)])
def test_staged_tables(pkg, ctx, workloads, case, M, K):
    u = CASES[case](workloads)
    amp, phase = weights(1, len(u))
    v = targets(2, M)
    y1, y0 = both(pkg, ctx, amp, phase, u, v, K, -1, obliquity=K < 1000)
    assert np.array_equal(y1, y0)
    ref = ctx.transform_mc(amp, phase, u, v, K, 7, -1, LAM, pkg.FP64, obliquity=K < 1000)
    assert rel_l2(y1, ref) <= 1e-6
