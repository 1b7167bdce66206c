"""A map copied out in the other precision goes through as large a device
buffer as can be had, and through the host where there is none: it does not
fail for want of device memory.  convert_out (p2m_convert.h) on the host
(tests/convert_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "matt_young_mapmaking_amd", "csrc")


def test_every_value_once_whatever_the_room(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not found")
    exe = tmp_path / "convert_check"
    subprocess.run([gxx, "-O1", "-std=c++17", "-I", CSRC, os.path.join(ROOT, "tests", "convert_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
    assert " 0 mismatches" in r.stdout
