"""Device memory kept for reuse (dmhm_amd/csrc/pool.hpp): its rules on a
counted host memory, and on the GPU that dmhm_trim gives it back."""
import os
import subprocess

import pytest

torch = pytest.importorskip("torch")        # before the library: both then share one HIP runtime
import dmhm_amd  # noqa: E402

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rules_on_a_counted_memory(tmp_path):
    exe = str(tmp_path / "block_pool")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I" + os.path.join(HERE, "..", "dmhm_amd", "csrc"),
                    os.path.join(HERE, "cpp", "block_pool.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout


@pytest.mark.gpu
def test_trim_gives_destroyed_matrices_back():
    dmhm_amd.init(0)
    free = lambda: torch.cuda.mem_get_info(0)[0]
    make = lambda: dmhm_amd.HMat2d.zeros([128, 128], 5, 16, True, dmhm_amd.DMHM_F64)
    make()                                  # its first use loads code
    dmhm_amd.trim()
    before = free()
    H = make()
    taken = before - free()
    assert taken > 1 << 27                  # a few hundred MB
    del H
    assert before - free() > taken // 2     # held for the next matrix
    dmhm_amd.trim()
    assert before - free() < taken // 2
