"""Monte Carlo draws up to K = 2^32 - 1: the arithmetic of their splits and of the
loops over a split, on the host (csrc/holo_mc.hpp as the kernels include it)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_splits_and_loops_up_to_the_largest_k(tmp_path):
    exe = str(tmp_path / "mc_draws")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I",
                    os.path.join(ROOT, "holographic-projector-simulations_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "mc_draws.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
