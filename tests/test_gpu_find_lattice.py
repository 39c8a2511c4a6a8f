"""FP32-split calls without a plan find and cut a lattice of sources on the device.
They have to give the bits of a plan, whose host builder cuts it, whatever the
sources are: lattices of every padding, followed by copies or other points, nearly
uniform ones, rows that fail late, and no lattice at all; and again after a call of
another size has left its buffers.
"""
import numpy as np
import pytest
import torch

from test_gpu_pairs import LAM, lattice, weights

pytestmark = pytest.mark.gpu


def edited(u, n, d, by):
    u = u.copy()
    u[n, d] += by
    return u


def sources(case, w):
    u = lattice(48, 40, 8e-6, -7e-6)
    return {
        "multiples of 16": lambda: lattice(64, 32, 8e-6, 8e-6),
        "multiples of 8": lambda: lattice(8, 72, 8e-6, 8e-6),
        "8 x 8": lambda: lattice(8, 8, 8e-6, 8e-6),
        "padded": lambda: lattice(33, 65, -8e-6, 7.5e-6),
        "odd tile columns": lambda: lattice(20, 144, 8e-6, 8e-6),
        "too thin": lambda: lattice(15, 30, 8e-6, 8e-6),
        "copies of source 0": lambda: w.reference_plane(1029, 5e-3, 0.0, 0.8),
        "other tail": lambda: np.concatenate([u, u[:7] + [1e-3, 2e-3, 1e-3]]),
        "tail too long": lambda: np.concatenate([u, u[:48] + [1e-3, 0, 0]]),
        "last row short": lambda: u[:-3],
        "row fails late": lambda: edited(u, 47 * 40 + 39, 1, 1e-9),
        "one z off": lambda: edited(u, 1000, 2, 1e-6),
        "uniform to 1e-10": lambda: edited(u, np.arange(40) + 400, 0, 8e-16),
        "uniform to 1e-8": lambda: edited(u, np.arange(40) + 400, 0, 8e-14),
        "one row": lambda: lattice(1, 300, 8e-6, 8e-6),
        "one column": lambda: lattice(300, 1, 8e-6, 8e-6),
        "cloud": lambda: np.random.default_rng(0).random((300, 3)) * 1e-3,
        "63 sources": lambda: lattice(9, 7, 8e-6, 8e-6),
    }[case]()


CASES = ["multiples of 16", "multiples of 8", "8 x 8", "padded", "odd tile columns", "too thin",
         "copies of source 0", "other tail", "tail too long", "last row short", "row fails late",
         "one z off", "uniform to 1e-10", "uniform to 1e-8", "one row", "one column", "cloud",
         "63 sources"]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("z, sign, obliquity", [(0.3, 1, False), (0.002, -1, True)])
def test_same_bits_as_a_plan(pkg, ctx, workloads, case, z, sign, obliquity):
    u = sources(case, workloads)
    v = lattice(24, 20, 8e-6, 7e-6, 1e-4, 0.0, z)
    amp, phase = weights(0, len(u))
    dev = [torch.tensor(a, device="cuda") for a in (amp, phase, u, v)]
    y = ctx.transform_full(*dev, sign, LAM, pkg.FP32_SPLIT, obliquity=obliquity).cpu().numpy()
    plan = ctx.plan(u)
    for off in (1, 0):  # the lattice-to-lattice kernel and the 16-row kernels
        pkg.set_option("grid_pairs", off)
        y = ctx.transform_full(*dev, sign, LAM, pkg.FP32_SPLIT, obliquity=obliquity).cpu().numpy()
        yp = plan.transform(amp, phase, v, sign, LAM, pkg.FP32_SPLIT, obliquity=obliquity)
        assert np.array_equal(y, yp)
    pkg.set_option("grid_pairs", 1)
    big = torch.tensor(lattice(80, 96, 5e-6, 5e-6), device="cuda")
    w = torch.ones(len(big), device="cuda", dtype=torch.float64)
    ctx.transform_full(w, w, big, dev[3], sign, LAM, pkg.FP32_SPLIT)
    again = ctx.transform_full(*dev, sign, LAM, pkg.FP32_SPLIT, obliquity=obliquity).cpu().numpy()
    pkg.set_option("grid_pairs", 0)
    last = ctx.transform_full(*dev, sign, LAM, pkg.FP32_SPLIT, obliquity=obliquity).cpu().numpy()
    pkg.set_option("grid_pairs", 1)
    assert np.array_equal(last, yp)
    assert np.array_equal(again, plan.transform(amp, phase, v, sign, LAM, pkg.FP32_SPLIT,
                                                obliquity=obliquity))
