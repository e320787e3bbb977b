"""What the kernels refine from the hardware's estimates (dmhm_amd/csrc/
refine.hpp), on the host with estimates off by 2^-23: within a few roundings of
long double, each bound the sum of the roundings on its way."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_refined_values_are_good_to_rounding(tmp_path):
    exe = str(tmp_path / "refine")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-ffp-contract=off",
                    "-I" + os.path.join(HERE, "..", "dmhm_amd", "csrc"), os.path.join(HERE, "cpp", "refine.cpp"),
                    "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
