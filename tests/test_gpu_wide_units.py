"""The 64-column units of the MFMA tile kernel, which phases of many wide tiles
take: H = U V^T imported exactly, H X and H^T X with hundreds of columns, and
the product of two such matrices (stacked factors read through the table),
against numpy in FP64. Last column chunks of 1, 49 and 64 columns, 16- and
32-row units."""
import numpy as np
import pytest

dmhm_amd = pytest.importorskip("dmhm_amd")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    dmhm_amd.init(0)
    yield


# 256 row atoms: eight or more column chunks make the 8,192 units.
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("sizes,levels,r,k", [((128, 128), 5, 8, 512), ((127, 125), 5, 17, 561), ((128, 128), 5, 5, 577)])
def test_many_columns(sizes, levels, r, k, prec):
    print("case", sizes, r, k, prec, flush=True)
    n = int(np.prod(sizes))
    rng = np.random.default_rng(n + r)
    dt = np.float64 if prec == "f64" else np.float32
    cut = lambda a: a.astype(dt).astype(np.float64)
    U, V, X = (cut(rng.standard_normal((n, c))) for c in (r, r, k))
    H = dmhm_amd.HMat2d.from_lowrank(sizes, levels, r, True, U, V,
                                     precision=dmhm_amd.DMHM_F64 if prec == "f64" else dmhm_amd.DMHM_F32)
    for mul, L, R in ((H.Multiply, U, V), (H.TransposeMultiply, V, U)):
        got = mul(0.5, X.astype(dt))
        ref = 0.5 * (L @ (R.T @ X))
        # Standard bound of nested sums: the leaves' entries, n + r + 4 roundings.
        bound = (n + r + 4) * np.finfo(dt).eps * 0.5 * (np.abs(L) @ (np.abs(R).T @ np.abs(X)))
        assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("sizes,r", [((128, 120), 12), ((96, 100), 20)])
def test_product_of_many_stacks(sizes, r):
    print("case", sizes, r, flush=True)
    n = int(np.prod(sizes))
    rng = np.random.default_rng(7 * n + r)
    U, V, S, T = (rng.standard_normal((n, r)) for _ in range(4))
    X = rng.standard_normal((n, 3))
    A = dmhm_amd.HMat2d.from_lowrank(sizes, 5, r, True, U, V)
    B = dmhm_amd.HMat2d.from_lowrank(sizes, 5, r, True, S, T)
    got = A.Multiply(2.0, B).Multiply(1.0, X)
    ref = 2.0 * (U @ ((V.T @ S) @ (T.T @ X)))
    scale = np.abs(U) @ (np.abs(V.T @ S) @ (np.abs(T.T) @ np.abs(X)))
    # n roundings through each product, and a factor 1000 for the conditioning
    # of a Gaussian sketch of r + 4 columns of a block of rank r.
    assert np.linalg.norm(got - ref) <= 1000 * n * np.finfo(float).eps * np.linalg.norm(2.0 * scale)
