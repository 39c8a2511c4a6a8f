"""NaN and infinities in the weights, sources and targets of HOLO_FP32_SPLIT calls
whose targets are on a lattice: every target that is not finite on the tiled and
16-row kernels (option "grid_pairs" = 0) is not finite with the option on, every
other one is, and infinities stay infinities where the tiled kernel gives them.
"""
import numpy as np
import pytest

from test_gpu_pairs import LAM, both, lattice, weights
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
