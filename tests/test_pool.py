"""Matrices shared between handles and threads (CPU): builds a small C++ driver
against spheresimulator_amd/csrc/pool.hpp and runs it."""
import os
import subprocess

from conftest import ROOT


def test_shared_matrices(tmp_path):
    csrc = os.path.join(ROOT, "spheresimulator_amd", "csrc")
    exe = str(tmp_path / "test_pool")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I" + csrc,
                    os.path.join(ROOT, "tests", "cpp", "test_pool.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
