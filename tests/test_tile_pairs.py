"""The tiles of bands and sectors and what the binning derives for a disc:
the rings it reaches, the tiles it may reach, and its pixel runs from the
chord relation, against the FP64 disc query on the host over random discs at
nside 1..8192 (tests/tile_pairs_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "matt_young_mapmaking_amd", "csrc")


def test_tiles_and_pairs_hold_every_run(tmp_path):
    hipcc = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")
    if not hipcc:
        pytest.skip("hipcc not found")
    exe = tmp_path / "tile_pairs_check"
    subprocess.run([hipcc, "-O2", "-std=c++17", "-x", "hip", "--offload-arch=gfx950", "-ffp-contract=off",
                    "-I", CSRC, os.path.join(ROOT, "tests", "tile_pairs_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
    assert " 0 mismatches" in r.stdout
