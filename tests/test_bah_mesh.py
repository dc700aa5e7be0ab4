"""The cluster tables of the bar-and-hinge kernel, checked on the CPU.

Compiles tests/bah_mesh_check.cpp against minim_amd/csrc/bah_mesh.hpp (the
header that the library builds its tables with) and runs it: every node owned
once, every element's energy counted once, every node's codes naming exactly
its elements in list order, every position and record within its table; for
sheets, nodes with more elements than a chunk holds, and degenerate lists.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_cluster_tables(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path / "bah_mesh_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-pthread", "-I", os.path.join(ROOT, "minim_amd", "csrc"),
                    os.path.join(HERE, "bah_mesh_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout[-2000:])
    assert r.returncode == 0, r.stdout[-2000:]
