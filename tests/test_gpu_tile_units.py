"""The MFMA tile kernel at the edges of its units: H = U V^T imported exactly,
H X and H^T X with more columns than the streaming kernels take, against
numpy in FP64. Ranks below, at and above the 8- and 16-wide inner chunks,
single rows and columns, and sizes on both sides of the rule that splits a
unit over four waves."""
import numpy as np
import pytest

dmhm_amd = pytest.importorskip("dmhm_amd")
pytestmark = pytest.mark.gpu

CASES = [  # sizes, levels, rank, columns
    ((3, 3), 2, 1, 9),           # boxes of 1 and 2 points
    ((9, 7), 3, 3, 17),
    ((16, 16), 3, 8, 16),
    ((33, 37), 3, 7, 33),        # leaves of 72 to 90 points: atoms of 64 and a remainder
    ((65, 34), 3, 17, 31),       # a 1-row remainder
    ((64, 64), 4, 8, 64),        # projections fill the chip: one wave per unit
    ((50, 41), 4, 12, 65),       # a second column chunk of one column
    ((13, 9, 11), 3, 20, 40),
]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_products_at_unit_edges(case, prec):
    sizes, levels, r, k = case
    n = int(np.prod(sizes))
    rng = np.random.default_rng(n + r)
    f64 = prec == "f64"
    dt = np.float64 if f64 else np.float32
    cut = lambda a: a.astype(dt).astype(np.float64)
    U, V, X, Y = (cut(rng.standard_normal((n, c))) for c in (r, r, k, k))
    cls = dmhm_amd.HMat2d if len(sizes) == 2 else dmhm_amd.HMat3d
    H = cls.from_lowrank(sizes, levels, max(r, 4), True, U, V,
                         precision=dmhm_amd.DMHM_F64 if f64 else dmhm_amd.DMHM_F32)
    eps = np.finfo(dt).eps
    prev = dmhm_amd.set_tile_engine("mfma")
    try:
        for op, L, R in (("N", U, V), ("T", V, U)):
            mul = H.Multiply if op == "N" else H.TransposeMultiply
            got = mul(0.5, X.astype(dt), -2.0, Y.astype(dt).copy(order="F"))
            ref = 0.5 * (L @ (R.T @ X)) - 2.0 * Y
            # Standard bound of nested sums: the leaves' entries, n + r + 4 roundings.
            bound = (n + r + 4) * eps * (0.5 * np.abs(L) @ (np.abs(R).T @ np.abs(X)) + 2.0 * np.abs(Y))
            assert np.all(np.abs(got - ref) <= bound), (op, float((np.abs(got - ref) / bound).max()))
    finally:
        dmhm_amd.set_tile_engine(prev)


@pytest.mark.parametrize("engine", ["mfma", "lds"])
@pytest.mark.parametrize("sizes,levels,r", [((16, 16), 3, 5), ((33, 37), 3, 12), ((50, 41), 4, 16), ((64, 64), 4, 20),
                                            ((13, 9, 11), 3, 7)])
def test_stacked_factors_read_through_the_table(sizes, levels, r, engine):
    """A B for A, B at full rank, whose low-rank terms are stacked: 64-column
    chunks of a stack start inside a factor when r does not divide 64."""
    n = int(np.prod(sizes))
    rng = np.random.default_rng(7 * n + r)
    U, V, S, T = (rng.standard_normal((n, r)) for _ in range(4))
    X = rng.standard_normal((n, 3))
    cls = dmhm_amd.HMat2d if len(sizes) == 2 else dmhm_amd.HMat3d
    A = cls.from_lowrank(sizes, levels, r, True, U, V)
    B = cls.from_lowrank(sizes, levels, r, True, S, T)
    prev = dmhm_amd.set_tile_engine(engine)
    try:
        got = A.Multiply(2.0, B).Multiply(1.0, X)
    finally:
        dmhm_amd.set_tile_engine(prev)
    ref = 2.0 * (U @ ((V.T @ S) @ (T.T @ X)))
    scale = np.abs(U) @ (np.abs(V.T @ S) @ (np.abs(T.T) @ np.abs(X)))
    # n roundings through each product, and a factor 1000 for the conditioning
    # of a Gaussian sketch of r + 4 columns of a block of rank r.
    assert np.linalg.norm(got - ref) <= 1000 * n * np.finfo(float).eps * np.linalg.norm(2.0 * scale)
