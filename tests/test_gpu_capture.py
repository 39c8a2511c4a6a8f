"""Calls captured into a HIP graph: a plan's first call needs no earlier one (its
scratch is the plan's, and it takes the splits that fit what the context has), and a
graph keeps the scratch it was captured with when later calls outgrow it.

Bars against the same call made eagerly: FP32-split 1e-6, FP64 1e-12 (the splits may
differ); bit for bit where the scratch was there.
"""
import numpy as np
import pytest

from test_gpu_pairs import LAM, lattice
from test_gpu_points import jittered

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def rel(a, b):
    return float((a - b).norm() / b.norm())


SOURCES = {"lattice": lambda: lattice(64, 64, 10e-6, 10e-6),
           "padded": lambda: lattice(30, 50, 10e-6, 10e-6),
           "jittered": lambda: jittered(40, 36, 10e-6)}
TARGETS = {"lattice": lambda: lattice(40, 48, 8e-6, 8e-6, z=0.3),
           "few": lambda: lattice(4, 4, 8e-6, 8e-6, z=0.3),
           "jittered": lambda: jittered(40, 48, 8e-6) + [0, 0, 0.3]}


def capture(call, side):
    import torch
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        y = call()
    return graph, y


@pytest.mark.parametrize("src", SOURCES)
@pytest.mark.parametrize("tgt", TARGETS)
@pytest.mark.parametrize("precision", [0, 1])
def test_a_plans_first_call(pkg, src, tgt, precision):
    import torch
    u, v = dev(SOURCES[src]()), dev(TARGETS[tgt]())
    n = len(u)
    g = torch.Generator(device="cuda").manual_seed(3)
    a, p = (torch.rand(n, dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ctx = pkg.Context(0, side.cuda_stream)
        plan = ctx.plan(u)
    call = lambda: plan.transform(a, p, v, 1, LAM, precision)
    graph, y = capture(call, side)
    for seed in (4, 5):  # new weights, eager work between the replays
        a.copy_(torch.rand(n, dtype=torch.float64, device="cuda", generator=g))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            ref = call()
        torch.cuda.synchronize()
        assert rel(y, ref) <= (1e-12 if precision == 0 else 1e-6)
    del graph
    plan.close()
    ctx.close()


@pytest.mark.parametrize("kind", ["plan", "full", "mc"])
def test_scratch_of_a_graph_outlives_its_growth(pkg, kind):
    """The captured call's splits lie in scratch that later eager calls outgrow."""
    import torch
    u, v = dev(SOURCES["lattice"]()), dev(TARGETS["lattice"]())
    big_u, big_v = dev(lattice(128, 96, 10e-6, 10e-6)), dev(lattice(250, 256, 8e-6, 8e-6, z=0.3))
    n = len(u)
    a, p = (torch.rand(k, dtype=torch.float64, device="cuda") for k in (n, n))
    ab, pb = (torch.rand(k, dtype=torch.float64, device="cuda") for k in (len(big_u),) * 2)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ctx = pkg.Context(0, side.cuda_stream)
        plan = ctx.plan(u)

        def call(a=a, p=p, u=u, v=v, plan=plan):
            if kind == "plan":
                return plan.transform(a, p, v, 1, LAM, pkg.FP32_SPLIT)
            if kind == "full":
                return ctx.transform_full(a, p, u, v, 1, LAM, pkg.FP64)
            return ctx.transform_mc(a, p, u, v, 700, 5, 1, LAM, pkg.FP32_SPLIT)

        ref = call()
    graph, y = capture(call, side)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, ref)
    with torch.cuda.stream(side):
        big = call(ab, pb, big_u, big_v, ctx.plan(big_u))
        again = call()
    torch.cuda.synchronize()
    assert torch.equal(again, ref) and torch.isfinite(torch.view_as_real(big)).all()
    junk = [torch.full((1 << 20,), float("nan"), dtype=torch.float64, device="cuda")
            for _ in range(8)]
    for _ in range(2):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
    assert all(torch.isnan(j).all() for j in junk)
    del graph
    plan.close()
    ctx.close()
