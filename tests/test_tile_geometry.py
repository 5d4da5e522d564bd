"""CPU check of the tile kernel's geometry (tests/tile_geometry_main.cpp, built with hipcc as host
code)."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_tile_geometry(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = tmp_path / "tile_geometry"
    subprocess.run([hipcc, "-O1", "-std=c++17", "-I", os.path.join(ROOT, "include"),
                    os.path.join(HERE, "tile_geometry_main.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True, timeout=600)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stderr
    assert "tile_geometry_main: ok" in res.stdout
