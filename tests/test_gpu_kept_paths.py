"""Calls beside the lattice-target kernels that keep a path of their own: product grids
that are not uniform (the 8 x 8 kernel), and calls without a plan, whose kept buffers
are written again on another stream.
"""
import numpy as np
import pytest

from test_gpu_pairs import LAM, both, lattice, rel_l2, weights
from test_gpu_points import jittered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [(20, 24), (70, 65)])
def test_nonuniform_product_grid(pkg, ctx, oracle, M):
    g = np.random.default_rng(8)
    x, y = np.cumsum(g.uniform(5e-6, 15e-6, 24)), np.cumsum(g.uniform(5e-6, 15e-6, 40))
    X, Y = np.meshgrid(x, y, indexing="ij")
    u, v = np.stack([X.ravel(), Y.ravel(), 0 * X.ravel()], 1), lattice(*M, 8e-6, 8e-6, z=0.25)
    plan = ctx.plan(u)
    assert plan.lattice() == (24, 40)
    amp, phase = weights(6, len(u))
    y1, y0 = both(pkg, lambda: plan.transform(amp, phase, v, 1, LAM, pkg.FP32_SPLIT))
    assert np.array_equal(y1, y0)
    assert rel_l2(y1, oracle.transform_full(1, LAM, amp, phase, u, v)) <= 1e-6


def test_calls_without_a_plan_on_two_streams(pkg):
    """Of several sizes and kinds of sources, in turn on two streams of one context;
    each with the bits that it has alone."""
    import torch
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    v = dev(lattice(48, 40, 8e-6, 8e-6, z=0.3))
    sources = [dev(a) for a in (lattice(96, 80, 9e-6, 9e-6), jittered(40, 36, 9e-6),
                                lattice(33, 50, 9e-6, 9e-6), lattice(128, 128, 9e-6, 9e-6),
                                jittered(90, 91, 9e-6), lattice(16, 16, 9e-6, 9e-6))]
    w = [tuple(torch.rand(len(u), dtype=torch.float64, device="cuda") for _ in range(2))
         for u in sources]

    def call(ctx, k):
        return ctx.transform_full(*w[k], sources[k], v, 1, LAM, pkg.FP32_SPLIT)

    alone = []
    for k in range(len(sources)):
        c = pkg.Context(0)
        alone.append(call(c, k))
        torch.cuda.synchronize()
        c.close()
    ctx, streams, got = pkg.Context(0), [torch.cuda.Stream() for _ in range(2)], []
    torch.cuda.synchronize()
    for r in range(3):
        for k in range(len(sources)):
            with torch.cuda.stream(streams[(k + r) % 2]):
                got.append((k, call(ctx, k)))
    torch.cuda.synchronize()
    assert all(torch.equal(y, alone[k]) for k, y in got)
    ctx.close()
