"""Which sphere pairs the right-hand side and the final velocities treat at the
sphere centres (CPU): builds a small C++ driver against
spheresimulator_amd/csrc/common.hpp and shtables.cpp and runs it."""
import os
import subprocess

from conftest import ROOT


def test_closed_forms_equal_the_grid_sums_where_they_replace_them(tmp_path):
    csrc = os.path.join(ROOT, "spheresimulator_amd", "csrc")
    exe = str(tmp_path / "test_centre_pairs")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__", "-I" + csrc,
                    os.path.join(ROOT, "tests", "cpp", "test_centre_pairs.cpp"), os.path.join(csrc, "shtables.cpp"),
                    "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    print(out.stdout)
    assert out.returncode == 0, out.stdout
