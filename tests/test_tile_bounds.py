"""Every pixel that a tile painter stores lies in its ring and the map, and
every map pixel belongs to one tile, at every nside and tile size, with the
shapes that the library builds (tests/tile_bounds_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "matt_young_mapmaking_amd", "csrc")


def test_tiles_cover_the_map_once(tmp_path):
    hipcc = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")
    if not hipcc:
        pytest.skip("hipcc not found")
    exe = tmp_path / "tile_bounds_check"
    subprocess.run([hipcc, "-O2", "-std=c++17", "-x", "hip", "--offload-arch=gfx950", "-ffp-contract=off",
                    "-I", CSRC, os.path.join(ROOT, "tests", "tile_bounds_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    assert " 0 mismatches" in r.stdout
