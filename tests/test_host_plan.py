"""How the engine plans and prepares a pass, on the CPU: a small C++ program
(tests/host_plan.cpp) linked against the library."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "gubingluo_amd")


def test_host_plan(tmp_path):
    if not os.path.exists(os.path.join(PKG, "librtm_hip.so")):
        pytest.fail("librtm_hip.so is not built")
    exe = str(tmp_path / "host_plan")
    cmd = ["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "include"),
           "-I", os.path.join(PKG, "csrc"), os.path.join(ROOT, "tests", "host_plan.cpp"), "-o", exe, "-L", PKG,
           "-lrtm_hip", f"-Wl,-rpath,{PKG}"]
    b = subprocess.run(cmd, capture_output=True, text=True)
    assert b.returncode == 0, b.stdout + b.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "all plan checks passed" in r.stdout
