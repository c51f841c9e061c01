"""The plans of FP32 triangles, checked on the CPU: tests/triangle_plan_check.cpp, built with hipcc against libmfx.so."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "sycl-bench_amd")
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_triangle_plans_are_the_estimated_ones(tmp_path):
    exe = str(tmp_path / "triangle_plan_check")
    b = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-I", os.path.join(PKG, "csrc"),
                        os.path.join(ROOT, "tests", "triangle_plan_check.cpp"), "-o", exe, "-L", PKG, "-lmfx",
                        "-Wl,-rpath," + PKG], capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    print(r.stdout, r.stderr[-3000:])
    assert r.returncode == 0 and r.stdout.startswith("OK")
