"""CPU check of the device blocks that adjoint runs keep (tests/kept_blocks_main.cpp, built with g++)."""
from __future__ import annotations

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_kept_blocks(tmp_path):
    exe = tmp_path / "kept_blocks"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread",
                    os.path.join(HERE, "kept_blocks_main.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True, timeout=300)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stderr
    assert "kept_blocks_main: ok" in res.stdout
