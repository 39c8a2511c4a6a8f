"""Calls that the C ABI refuses before anything is queued on the device."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("missing", ["amp", "phase", "u", "v", "y"])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("N", [1, 64, 300])
def test_transform_full_device_null_array(pkg, ctx, missing, precision, N):
    import torch
    M = 300
    t = {k: torch.zeros(n, dtype=torch.float64, device="cuda")
         for k, n in (("amp", N), ("phase", N), ("u", 3 * N), ("v", 3 * M), ("y", 2 * M))}
    p = {k: None if k == missing else ctypes.c_void_p(a.data_ptr()) for k, a in t.items()}
    status = pkg.lib().holo_transform_full(ctx.handle, precision, 1, 632.8e-9, p["amp"],
                                           p["phase"], p["u"], N, p["v"], M, p["y"], None,
                                           pkg.DEVICE_POINTERS)
    assert status == 1 and b"null" in pkg.lib().holo_last_error()
