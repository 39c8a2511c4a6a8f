"""holo_trim: the scratch that calls keep is given back, and the calls after it give
the bits of the calls before."""
import numpy as np
import pytest

from test_gpu_pairs import LAM, lattice

pytestmark = pytest.mark.gpu


def test_trim_frees_what_calls_keep(pkg):
    import torch
    free = lambda: torch.cuda.mem_get_info()[0]
    u = torch.from_numpy(lattice(512, 512, 10e-6, 10e-6)).cuda()
    v = torch.from_numpy(lattice(300, 300, 8e-6, 8e-6, z=0.3)).cuda()
    a, p = (torch.rand(len(u), dtype=torch.float64, device="cuda") for _ in range(2))
    c = pkg.Context(0)

    def calls():
        return [c.transform_full(a, p, u, v, 1, LAM, pkg.FP32_SPLIT),
                c.transform_full(a, p, u, v, 1, LAM, pkg.FP64),
                c.transform_mc(a, p, u, v, 64, 3, 1, LAM, pkg.FP32_SPLIT)]

    c.trim()  # nothing there
    before = calls()
    torch.cuda.synchronize()
    held = free()
    c.trim()
    freed = free() - held
    print(f"{freed / 2**20:.0f} MiB given back")
    assert freed >= 16 * 2**20  # the plan of 2^18 sources alone is some 30 MB
    for _ in range(2):
        assert all(torch.equal(x, y) for x, y in zip(calls(), before))
        c.trim()
    c.close()
