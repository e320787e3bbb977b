"""The MFMA tile kernel's walk over the inner chunks of a tile's contributions
(dmhm_amd/csrc/chunks.hpp), replayed on the host for all pairs and triples of
inner dimensions up to 256: no fetch, the repeated last one included, leaves
the contribution whose operands are set, and every chunk is taken once."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_fetch_lies_inside_its_contribution(tmp_path):
    exe = str(tmp_path / "chunk_walk")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I" + os.path.join(HERE, "..", "dmhm_amd", "csrc"),
                    os.path.join(HERE, "cpp", "chunk_walk.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
