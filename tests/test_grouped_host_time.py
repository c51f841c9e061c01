"""Host time of choosing a grouped launch's policy (CPU): tests/grouped_host_time.cpp, built with hipcc against
libmfx.so, plans lists with and without a given policy."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "sycl-bench_amd")
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_choosing_a_policy_costs_little_more_than_planning_it(tmp_path):
    exe = str(tmp_path / "grouped_host_time")
    b = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-I", os.path.join(PKG, "csrc"),
                        os.path.join(ROOT, "tests", "grouped_host_time.cpp"), "-o", exe, "-L", PKG, "-lmfx",
                        "-Wl,-rpath," + PKG], capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    print(r.stdout, r.stderr[-3000:])
    assert r.returncode == 0 and r.stdout.endswith("OK\n")
