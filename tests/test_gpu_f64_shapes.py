"""FP64 launches over the sizes where their shape (targets per lane, source
splits) and the device's layout scan change: against the oracle (<= 1e-12), and
device positions (layout found on the GPU) against host positions (scanned on
the host), bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAM = 632.8e-9


def rel_l2(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def sources(kind, n):
    g = np.random.default_rng(n)
    u = (g.random((n, 3)) - 0.5) * 2e-3
    if kind != "cloud":
        u[:, 2] = 0.0
    if kind == "rows":  # rows of 37 with one x, the last one short
        u[:, 0] = np.repeat((g.random(-(-n // 37)) - 0.5) * 2e-3, 37)[:n]
    return u


@pytest.mark.parametrize("kind", ["cloud", "plane", "rows"])
@pytest.mark.parametrize("n, m", [(1, 1), (3, 257), (31, 256), (64, 255), (65, 1025), (1000, 300),
                                  (8192, 40), (8193, 40), (4100, 700)])
def test_shapes(pkg, ctx, oracle, kind, n, m):
    import torch
    u = sources(kind, n)
    g = np.random.default_rng(m)
    v = np.concatenate([(g.random((m, 2)) - 0.5) * 4e-3, np.full((m, 1), 0.3)], 1)
    amp, phase = g.random(n), g.random(n) * 2 * np.pi
    host = ctx.transform_full(amp, phase, u, v, -1, LAM, pkg.FP64)
    dev = ctx.transform_full(*[torch.from_numpy(a).cuda() for a in (amp, phase, u, v)], -1, LAM,
                             pkg.FP64).cpu().numpy()
    ref = oracle.transform_full(-1, LAM, amp, phase, u, v)
    assert rel_l2(host, ref) <= 1e-12
    assert np.array_equal(host, dev)
