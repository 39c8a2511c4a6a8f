"""NaN and infinities in the weights, sources and targets of HOLO_FP32_SPLIT calls
whose targets are on a lattice: every target that is not finite on the tiled and
16-row kernels (option "grid_pairs" = 0) is not finite with the option on, every
other one is, and infinities stay infinities where the tiled kernel gives them.
Wavelengths and lengths at the ends of what FP32 holds: within 1e-6 of the oracle.
"""
import numpy as np
import pytest

from test_gpu_pairs import LAM, both, lattice, rel_l2, weights
from test_gpu_points import jittered

pytestmark = pytest.mark.gpu


def kinds(y):
    z = y.view(np.float64)
    return np.where(np.isnan(z), 2, np.where(np.isinf(z), np.sign(z), 0))


@pytest.mark.parametrize("where", ["amp", "phase", "source x", "source z", "target y", "target z"])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("z", [0.3, 0.08])
def test_nonfinite_inputs(pkg, ctx, where, value, z):
    v = lattice(33, 40, 8e-6, 8e-6, z=z)
    for on_lattice, u in ((True, lattice(40, 36, 9e-6, 8e-6)), (False, jittered(40, 36, 9e-6))):
        amp, phase = weights(3, len(u))
        w, k = v.copy(), 700
        if where == "amp":
            amp[k] = value
        elif where == "phase":
            phase[k] = value
        elif where.startswith("source"):
            u[k, "xyz".index(where[-1])] = value
        else:
            w[k, "xyz".index(where[-1])] = value
        plan = ctx.plan(u)
        y1, y0 = both(pkg, lambda: plan.transform(amp, phase, w, 1, LAM, pkg.FP32_SPLIT))
        assert not np.isfinite(y0).all()
        assert np.array_equal(np.isfinite(y1), np.isfinite(y0))
        if not on_lattice:
            assert np.array_equal(kinds(y1), kinds(y0))


@pytest.mark.parametrize("value", [np.nan, np.inf, 1e39, 1e39j, complex(0, np.nan)])
def test_nonfinite_complex_weights(pkg, ctx, value):
    """Complex weights, 1e39 among them: an infinity in FP32."""
    v = lattice(33, 40, 8e-6, 8e-6, z=0.3)
    for u in (lattice(40, 36, 9e-6, 8e-6), jittered(40, 36, 9e-6)):
        w = np.exp(1j * np.arange(len(u)))
        w[300] = value
        plan = ctx.plan(u)
        y1, y0 = both(pkg, lambda: plan.transform_complex(w, v, -1, LAM, pkg.FP32_SPLIT))
        assert not np.isfinite(y0).all()
        assert np.array_equal(np.isfinite(y1), np.isfinite(y0))


def test_all_targets_at_infinite_distance(pkg, ctx):
    v = lattice(33, 40, 8e-6, 8e-6, z=np.inf)
    for u in (lattice(40, 36, 9e-6, 8e-6), jittered(40, 36, 9e-6)):
        plan = ctx.plan(u)
        amp, phase = weights(4, len(u))
        y1, y0 = both(pkg, lambda: plan.transform(amp, phase, v, 1, LAM, pkg.FP32_SPLIT))
        assert np.array_equal(np.isfinite(y1), np.isfinite(y0))


@pytest.mark.parametrize("lam", [1e-12, 1e-3, 1.0, 1e20, 1e30, 1e33, 1e38, 1e100, 1e300])
def test_wavelengths_at_the_ends_of_the_range(pkg, ctx, oracle, lam):
    """Every wavelength that FP32 sums take; where a phase per FP32 unit is too small for
    the lattice-target kernels' scales the others keep the call."""
    v = lattice(33, 40, 8e-6, 8e-6, z=0.3)
    for u in (lattice(40, 36, 9e-6, 8e-6), jittered(40, 36, 9e-6)):
        amp, phase = weights(5, len(u))
        y = ctx.plan(u).transform(amp, phase, v, 1, lam, pkg.FP32_SPLIT)
        ref = oracle.transform_full(1, lam, amp, phase, u, v)
        # (1e-12 m: 3e11 cycles, 2e-4 by FP64 rounding alone)
        assert rel_l2(y, ref) <= (1e-6 if lam > 1e-6 else 1e-3)


@pytest.mark.parametrize("scale", [1e-12, 1e-9, 1e-6, 1e-3, 1e3, 1e6, 1e8, 1e9, 1e10, 1e12])
@pytest.mark.parametrize("z", [0.3, 0.05])
def test_scales_of_lengths(pkg, ctx, oracle, scale, z):
    """The same geometry in other units."""
    v = lattice(33, 40, 20e-6, 8e-6, 1e-3, z=z) * scale
    for u in (lattice(40, 36, 9e-6, 8e-6), jittered(40, 36, 9e-6)):
        amp, phase = weights(5, len(u))
        y = ctx.plan(u * scale).transform(amp, phase, v, 1, LAM * scale, pkg.FP32_SPLIT)
        ref = oracle.transform_full(1, LAM * scale, amp, phase, u * scale, v)
        assert rel_l2(y, ref) <= 1e-6
