"""Host-only checks of the planner's inner rules (no GPU): tests/planner/planner_check.cpp, compiled with the library's host source."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


def test_planner_rules(tmp_path):
    if not (os.path.exists(HIPCC) or shutil.which(HIPCC)):
        pytest.skip("hipcc not available")
    lib = os.path.join(ROOT, "flashfftstencil_amd")
    exe = str(tmp_path / "planner_check")
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-mcode-object-version=5", "-O2", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", os.path.join(ROOT, "tests", "planner", "planner_check.cpp"), f"-L{lib}",
                        "-lffstencil", f"-Wl,-rpath,{lib}", "-o", exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "planner checks passed" in r.stdout, r.stdout + r.stderr
