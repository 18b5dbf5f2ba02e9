"""Accuracy of the far-field levels (CPU): builds a small C++ driver against
spheresimulator_amd/csrc/shtables.cpp and runs it."""
import os
import subprocess

from conftest import ROOT


def test_levels_are_no_further_off_than_gauss_legendre_grids(tmp_path):
    csrc = os.path.join(ROOT, "spheresimulator_amd", "csrc")
    exe = str(tmp_path / "test_level_errors")
    subprocess.run(["g++", "-O3", "-std=c++17", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__", "-I" + csrc,
                    os.path.join(ROOT, "tests", "cpp", "test_level_errors.cpp"), os.path.join(csrc, "shtables.cpp"),
                    "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
