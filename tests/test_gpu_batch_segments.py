"""Batched products on the engine that callers get (segmented MFMA launches):
members U_i V_i^T and S_i T_i^T imported exactly at full rank, whose stacked
terms are read through each member's own table, against numpy. Batches below
the four-wave split's line of units, above it and above that of the 64-column
units; more than 64 members; two classes in one batch. Entries are positive,
so nothing cancels: each row of C_i x_i within 100 sqrt(n) roundings (sums of
up to n terms, rounding errors added at random, and a sketch of r + 4 columns
of a block of rank r)."""
import numpy as np
import pytest

import dmhm_amd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    dmhm_amd.init(0)
    yield


BATCHES = [  # (sizes, levels, rank, members) per class
    [((16, 16), 3, 5, 3)],
    [((16, 16), 3, 3, 70)],
    [((33, 37), 3, 12, 4)],
    [((48, 48), 4, 8, 12)],
    [((64, 60), 4, 8, 24)],
    [((50, 41), 4, 20, 5)],
    [((13, 9, 11), 3, 7, 6)],
    [((16, 16), 3, 8, 5), ((24, 20), 3, 8, 4)],
]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("classes", BATCHES, ids=[str(b) for b in BATCHES])
def test_batched_products_of_exact_members(classes, prec):
    dt = np.float64 if prec == "f64" else np.float32
    code = dmhm_amd.DMHM_F64 if prec == "f64" else dmhm_amd.DMHM_F32
    As, Bs, facs = [], [], []
    for sizes, levels, r, count in classes:
        n = int(np.prod(sizes))
        cls = dmhm_amd.HMat2d if len(sizes) == 2 else dmhm_amd.HMat3d
        for i in range(count):
            rng = np.random.default_rng(1000 * n + i)
            U, V, S, T = (rng.uniform(0.5, 1.5, (n, r)).astype(dt).astype(np.float64) for _ in range(4))
            As.append(cls.from_lowrank(sizes, levels, r, True, U, V, precision=code))
            Bs.append(cls.from_lowrank(sizes, levels, r, True, S, T, precision=code))
            facs.append((U, V, S, T, rng.uniform(0.5, 1.5, (n, 2)).astype(dt)))
    prev = dmhm_amd.set_tile_engine("auto")
    try:
        C = dmhm_amd.HBatch.create(As).Multiply(2.0, dmhm_amd.HBatch.create(Bs))
    finally:
        dmhm_amd.set_tile_engine(prev)
    for i, (U, V, S, T, x) in enumerate(facs):
        got = C.member(i).Multiply(1.0, x)
        want = 2.0 * (U @ ((V.T @ S) @ (T.T @ x.astype(np.float64))))
        assert np.all(np.abs(got - want) <= 100 * np.sqrt(len(U)) * np.finfo(dt).eps * want), i
