"""CPU test of the rules that choose between the multi-rhs hopping kernels (tile_rhs and split_rhs
in wl_internal.h): tests/cpp/test_tile_rules.hip is compiled host-only with hipcc and run."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or ("/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else None)


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc")
def test_rules_take_the_kernel_that_was_measured_faster(tmp_path):
    exe = tmp_path / "test_tile_rules"
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "hila_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_tile_rules.hip"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr
    assert "rules ok" in p.stdout
