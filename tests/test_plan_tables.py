"""The tables of a product's plan, lowered on the host: stacked factors are read
through one entry per factor and one per stack, not per column, and every entry
leads to a stored factor's columns."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "dmhm_amd", "csrc")


def test_stacks_are_read_through_small_tables(tmp_path):
    exe = str(tmp_path / "plan_tables")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + CSRC, os.path.join(HERE, "cpp", "plan_tables.cpp"),
                    os.path.join(CSRC, "plan.cpp"), os.path.join(CSRC, "geometry.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
