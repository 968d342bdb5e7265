"""CPU test of the tiles of the direction-split hopping kernel (split_geom in wl_internal.h,
split_site in wl_split.h): tests/cpp/test_split_cover.hip is compiled host-only with hipcc and run
over lattices whose extents are small, odd multiples of two, one row wide or too wide to tile."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or ("/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else None)


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc")
def test_tiles_cover_the_lattice_and_stage_the_neighbours(tmp_path):
    exe = tmp_path / "test_split_cover"
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "hila_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_split_cover.hip"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr
    assert "cover ok" in p.stdout
