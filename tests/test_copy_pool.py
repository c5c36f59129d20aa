"""The host copy pool's constructor where memory runs out part way: the threads
that could be started, or the caller alone, copy the rows (CPU only)."""
from __future__ import annotations

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
HOST = os.path.join(HERE, "..", "p2z-tests_amd", "host")


def test_construction_out_of_memory(tmp_path):
    exe = str(tmp_path / "copy_pool_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", HOST, os.path.join(HOST, "p2z_copy.cpp"),
                    os.path.join(HERE, "copy_pool_check.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, (run.returncode, run.stdout, run.stderr)
