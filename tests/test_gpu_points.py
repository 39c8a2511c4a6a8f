"""The point-to-lattice kernel (HOLO_FP32_SPLIT, sources off a uniform lattice,
targets on one) at the edges of its batches, tiles and forms.

Bar: relative L2 <= 1e-6 against the FP64 oracle, as for every FP32-split path.
Option "grid_pairs" = 0 keeps such calls on the tiled and 8 x 8 kernels; calls
whose targets are no lattice, or whose plan asks for another tile, give the same
bits with the option on and off.
"""
import numpy as np
import pytest

from test_gpu_pairs import LAM, both, lattice, rel_l2, weights

pytestmark = pytest.mark.gpu


def jittered(nx, ny, p, seed=0, depth=0.0):
    u = lattice(nx, ny, p, p)
    g = np.random.default_rng(seed)
    u[:, :2] += (g.random((len(u), 2)) - 0.5) * 0.975 * p
    u[:, 2] += (g.random(len(u)) - 0.5) * depth
    return u


def check(pkg, ctx, oracle, u, v, sign=1, obliquity=False, seed=0, other=True, tile=64, scale=1.0):
    amp, phase = weights(seed, len(u))
    plan = ctx.plan(u, tile)
    y1, y0 = both(pkg, lambda: plan.transform(amp * scale, phase, v, sign, LAM, pkg.FP32_SPLIT,
                                              obliquity=obliquity) / scale)
    ref = oracle.transform_full(sign, LAM, amp, phase, u, v, obliquity=obliquity)
    print(f"rel L2 {rel_l2(y1, ref):.2e} (tiled kernel {rel_l2(y0, ref):.2e})")
    assert rel_l2(y1, ref) <= 1e-6
    assert np.array_equal(y1, y0) != other


@pytest.mark.parametrize("n", [255, 256, 257, 271, 272, 273, 319, 320, 321, 1100])
@pytest.mark.parametrize("tgt", [(16, 16), (16, 33), (33, 65)])
def test_batch_and_tile_edges(pkg, ctx, oracle, n, tgt):
    g = np.random.default_rng(n)
    u = (g.random((n, 3)) - 0.5) * [2e-3, 2e-3, 1e-2]
    check(pkg, ctx, oracle, u, lattice(*tgt, 7e-6, -7.56e-6, 1e-4, z=0.3), other=n >= 256)


# far form, near form, and beyond (the tiled kernel, bit for bit)
@pytest.mark.parametrize("z, other", [(0.35, True), (0.1, True), (0.05, True), (0.015, False)])
@pytest.mark.parametrize("sign, obliquity", [(1, False), (-1, True)])
def test_forms(pkg, ctx, oracle, z, other, sign, obliquity):
    check(pkg, ctx, oracle, jittered(48, 60, 20e-6), lattice(40, 48, 20e-6, 15e-6, 5e-4, -5e-4, z),
          sign, obliquity, other=other)


def test_one_source_far_before_the_others(pkg, ctx, oracle):
    """Amplitudes a hundredth of the nearest source's still carry the field."""
    u = jittered(64, 64, 10e-6, 6, 0.2)
    u[:, 2] -= 1.0
    u[5] = [1e-4, 0, 0]
    check(pkg, ctx, oracle, u, lattice(40, 48, 8e-6, 8e-6, z=0.02))


@pytest.mark.parametrize("splits", [0, 1, 3])
@pytest.mark.parametrize("scale", [1e-30, 1.0, 1e25])
def test_splits_scales_and_target_copies(pkg, ctx, oracle, workloads, splits, scale):
    pkg.set_option("splits", splits)
    check(pkg, ctx, oracle, jittered(40, 30, 10e-6, 1, 2e-3),
          workloads.reference_plane(1029, 5e-4, 0.3, 0.8), -1, scale=scale)
    pkg.set_option("splits", 0)


def test_other_paths_keep_theirs(pkg, ctx, oracle):
    """Targets off a lattice, a plan with another tile, targets among the sources."""
    u = jittered(40, 30, 10e-6, 2)
    v = lattice(20, 24, 8e-6, 8e-6, z=0.3)
    w = v.copy()
    w[77, 1] += 1e-9
    check(pkg, ctx, oracle, u, w, other=False)
    check(pkg, ctx, oracle, u, v, other=False, tile=16)
    deep = u + np.array([0, 0, 1e-3]) * np.linspace(-1, 1, len(u))[:, None]
    check(pkg, ctx, oracle, deep, lattice(20, 24, 8e-6, 8e-6, z=5e-4), other=False)


def test_nonuniform_product_grid_and_complex_adjoint(pkg, ctx, oracle):
    """A product grid that is not uniform (the 8 x 8 kernel's) keeps that kernel;
    complex weights and the adjoint of jittered targets take this one."""
    g = np.random.default_rng(3)
    u, v = jittered(30, 20, 10e-6, 4), lattice(24, 30, 9e-6, 8e-6, z=0.25)
    w = g.standard_normal(len(u)) + 1j * g.standard_normal(len(u))
    w[100:200] = 0.0
    y1, y0 = both(pkg, lambda: ctx.plan(u).transform_complex(w, v, -1, LAM, pkg.FP32_SPLIT))
    assert rel_l2(y1, oracle.transform_cartesian(-1, LAM, w, u, v)) <= 1e-6
    assert not np.array_equal(y1, y0)
    amp, theta = weights(5, len(v))
    ga, gt = ctx.plan(u).adjoint(w, amp, theta, v, +1, LAM, pkg.FP32_SPLIT)
    ra, rt = oracle.adjoint(+1, LAM, amp, theta, v, w, u)
    assert rel_l2(ga, ra) <= 1e-6 and rel_l2(gt, rt) <= 1e-6
