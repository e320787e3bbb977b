"""Repeated calls on the default tile engine give the same bits: a direct
inversion (its program and arena stay with the geometry between calls) with
calls on another geometry between, and a batched product."""
import numpy as np
import pytest

import dmhm_amd
from dmhm_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    dmhm_amd.init(0)
    prev = dmhm_amd.set_tile_engine("auto")
    yield
    dmhm_amd.set_tile_engine(prev)


def operand(n, seed):
    op = W.small_operator(n, 3, smooth=False, seed=seed)
    return dmhm_amd.HMat2d.from_csr(op["sizes"], 3, 8, True, op["rowptr"], op["colind"], op["vals"])


def test_direct_inversions():
    A, B = operand(16, 5), operand(12, 6)
    inverse = lambda H: H.Copy().DirectInvert().to_dense()
    a, b = inverse(A), inverse(B)
    for _ in range(4):
        assert np.array_equal(inverse(A), a)
        assert np.array_equal(inverse(B), b)


def test_batched_products():
    hs = [operand(16, s).DirectInvert() for s in range(5)]
    batch = dmhm_amd.HBatch.create(hs)
    product = lambda: [batch.Multiply(1.0, batch, seed=3).member(i).to_dense() for i in range(5)]
    first = product()
    for _ in range(3):
        assert all(np.array_equal(x, y) for x, y in zip(product(), first))
