"""Device memory kept for reuse (dmhm_amd/csrc/pool.hpp): its rules on a
counted host memory."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rules_on_a_counted_memory(tmp_path):
    exe = str(tmp_path / "block_pool")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I" + os.path.join(HERE, "..", "dmhm_amd", "csrc"),
                    os.path.join(HERE, "cpp", "block_pool.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout

