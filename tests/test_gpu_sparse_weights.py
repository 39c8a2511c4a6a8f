"""The lattice-to-lattice kernel's forms with few lit sources.  Over dense weights the
terms a form drops average out over a tile; one lit source in a tile's corner leaves
each target the largest of them.

Bar: 1e-6, as for every FP32-split path, of the field or (where the sources cancel) of
the root of the sum of the squares of what they give alone.  Expected: the bounds of
the forms leave at most 2.5e-7 (far) and 1.4e-7 (near), the f16 parts of the small
products about 2e-7 and 4e-7 over the targets, the rest of the arithmetic 2e-7.
"""
import numpy as np
import pytest

from test_gpu_pairs import LAM, lattice

pytestmark = pytest.mark.gpu

# sides, pitches and offset: coarse sources and fine targets far off the axis (the
# largest share of a tile pair's cross term in every pair), and comparable pitches
GEOMETRIES = {
    "64 x 64 at 20 um, targets at 0.5 um": ((64, 64), (20e-6, 20e-6), (32, 32), (0.5e-6, 0.5e-6),
                                            (5.8e-3, 4e-3)),
    "128 x 256 at 10 um, targets at 1 um": ((128, 256), (10e-6, 10e-6), (32, 64), (1e-6, 1e-6),
                                            (2e-3, 2e-3)),
    "32 x 32 at 15 um, targets at 12 um": ((32, 32), (15e-6, 12e-6), (64, 40), (12e-6, 9e-6),
                                           (-3e-3, 1e-3)),
    "160 x 320 at 8 um, targets at 8 um": ((160, 320), (8e-6, 8e-6), (96, 96), (8e-6, 8e-6),
                                           (0.0, 0.0)),
}


def plane(geometry, cross):
    """Sources, and targets at the distance where narrow source tiles have this cross
    at the pair of tiles furthest off the axis."""
    src, sp, tgt, tp, off = geometry

    def reach(n, p, m, q, o):
        s = -(n - 1) / 2 * p + 15.5 * p + np.arange(-(-n // 32)) * 32 * p
        t = o - (m - 1) / 2 * q + 15.5 * q + np.arange(-(-m // 32)) * 32 * q
        r, h = np.abs(t[:, None] - s).max(), 15.5 * (p + q)
        return 2 * r * h + h * h

    pq = reach(src[0], sp[0], tgt[0], tp[0], off[0]) * reach(src[1], sp[1], tgt[1], tp[1], off[1])
    z = (np.pi / 2 * pq / (LAM * cross)) ** (1 / 3)
    return lattice(*src, *sp), lattice(*tgt, *tp, *off, z)


@pytest.mark.parametrize("geometry", GEOMETRIES)
@pytest.mark.parametrize("cross", [0.9e-3, 1.1e-3, 2.3e-3, 0.02, 0.055, 0.11])
@pytest.mark.parametrize("lit", ["corner", "one per tile", "four"])
@pytest.mark.parametrize("sign, obliquity", [(1, False), (-1, True)])
def test_few_lit_sources(pkg, ctx, oracle, geometry, cross, lit, sign, obliquity):
    geo = GEOMETRIES[geometry]
    u, v = plane(geo, cross)
    (nx, ny), off = geo[0], geo[4]
    # the corner that is furthest from the targets
    i, j = (0 if off[0] >= 0 else nx - 1), (0 if off[1] >= 0 else ny - 1)
    g = np.random.default_rng(11)
    w = np.zeros((nx, ny))
    if lit == "corner":
        w[i, j] = 1.0
    elif lit == "one per tile":
        w[i % 32::32, j % 64::64] = 1.0
    else:
        w[g.integers(0, nx, 4), g.integers(0, ny, 4)] = 1.0
    amp, phase = w.ravel(), g.random(nx * ny) * 2 * np.pi
    y = ctx.plan(u).transform(amp, phase, v, sign, LAM, pkg.FP32_SPLIT, obliquity=obliquity)
    k = np.flatnonzero(amp)
    ref = oracle.transform_full(sign, LAM, amp[k], phase[k], u[k], v, obliquity=obliquity)
    d = np.linalg.norm(v[:, None] - u[None, k], axis=2)
    alone = np.sqrt((((np.abs(v[:, None, 2] - u[None, k, 2]) / d if obliquity else 1) / d) ** 2).sum())
    err = np.linalg.norm(y - ref)
    print(f"{err / np.linalg.norm(ref):.2e} of the field, {err / alone:.2e} of the sources alone")
    assert err <= 1e-6 * max(np.linalg.norm(ref), alone)


@pytest.mark.parametrize("scale", [1e-38, 1e-30, 1.0, 1e30])
@pytest.mark.parametrize("src", [(16, 16), (33, 65), (64, 96)])
def test_polar_weights_of_any_scale(pkg, ctx, oracle, scale, src):
    """Amplitudes (of either sign) whose tiles differ by 1e6, and tiles of zeros: a tile's
    scale comes from its largest modulus."""
    u, v = lattice(*src, 10e-6, 9e-6), lattice(33, 44, 8e-6, 8e-6, 5e-4, 0, 0.3)
    g = np.random.default_rng(5)
    a = g.standard_normal(src)
    a[32:] *= 1e-6
    a[:, 64:] = 0.0
    amp, phase = a.ravel(), g.random(a.size) * 2 * np.pi
    y = ctx.plan(u).transform(amp * scale, phase, v, 1, LAM, pkg.FP32_SPLIT) / scale
    ref = oracle.transform_full(1, LAM, amp, phase, u, v)
    assert np.linalg.norm(y - ref) <= 1e-6 * np.linalg.norm(ref)
