"""The untuned choice of a grouped launch, checked on the CPU: tests/grouped_choice_check.cpp, built with hipcc against
libmfx.so."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "sycl-bench_amd")
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_packed_problems_beside_a_chain_leave_its_policy(tmp_path):
    exe = str(tmp_path / "grouped_choice_check")
    b = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-I", os.path.join(PKG, "csrc"),
                        os.path.join(ROOT, "tests", "grouped_choice_check.cpp"), "-o", exe, "-L", PKG, "-lmfx",
                        "-Wl,-rpath," + PKG], capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    print(r.stdout, r.stderr[-3000:])
    assert r.returncode == 0 and r.stdout.startswith("OK")
