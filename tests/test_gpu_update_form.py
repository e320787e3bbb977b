"""The update form C := alpha A B + beta C in place: against numpy where no
block is truncated (rank(A B) + rank(C) at most maxRank), with C's subtrees cut
into one workspace batch each, and with C as an operand. FP64, 1e-11 relative
to the entries summed: n roundings per product and the conditioning of a
Gaussian sketch with four columns to spare."""
import os
import subprocess
import sys

import numpy as np
import pytest

import dmhm_amd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    dmhm_amd.init(0)
    yield


CASES = [((16, 16), 3, True), ((50, 41), 4, True), ((33, 37), 3, False), ((13, 9, 11), 3, True)]


def operand(sizes, levels, strong, seed, r):
    n = int(np.prod(sizes))
    rng = np.random.default_rng(n + seed)
    U, V = rng.standard_normal((n, r)), rng.standard_normal((n, r))
    cls = dmhm_amd.HMat2d if len(sizes) == 2 else dmhm_amd.HMat3d
    return cls.from_lowrank(sizes, levels, 12, strong, U, V), U @ V.T


def close(got, want, terms):
    return np.abs(got - want).max() <= 1e-11 * terms.max()


def check_update(sizes, levels, strong):
    (A, a), (B, b), (C, c) = (operand(sizes, levels, strong, s, 4) for s in range(3))
    C.UpdateWith(0.0, C.Copy())             # standard layout, as products have
    A.Multiply(-0.5, B, 2.0, C)
    assert close(C.to_dense(), -0.5 * a @ b + 2.0 * c, np.abs(a) @ np.abs(b) + np.abs(c)), (sizes, strong)


@pytest.mark.parametrize("which", ["A", "B", "AB"])
@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_operand_is_the_result(case, which):
    (A, a), (C, c) = (operand(*case, s, 4) for s in range(2))
    C.UpdateWith(0.0, C.Copy())
    L, l = (C, c) if "A" in which else (A, a)
    R, r = (C, c) if "B" in which else (A, a)
    L.Multiply(-0.5, R, 2.0, C)
    assert close(C.to_dense(), -0.5 * l @ r + 2.0 * c, np.abs(l) @ np.abs(r) + np.abs(c))


def test_one_batch_per_subtree():
    # The budget is read once per process.
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, DMHM_HH_BATCH_ELEMS="1", PYTHONPATH=root)
    subprocess.run([sys.executable, os.path.abspath(__file__)], env=env, check=True, timeout=100)


if __name__ == "__main__":
    dmhm_amd.init(0)
    for case in CASES:
        check_update(*case)
