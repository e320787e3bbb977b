"""H X and H^T X with 1 to 8 columns against numpy in FP64: H = U V^T imported
exactly, on boxes below and above the size where a projection takes a
workgroup, ragged leaves and atoms, ranks on both sides of a 16-column record,
weak admissibility, every number of waves per atom, and device operands that
are misaligned and strided."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")        # before the library: both then share one HIP runtime
dmhm_amd = pytest.importorskip("dmhm_amd")
pytestmark = pytest.mark.gpu

CASES = [  # sizes, levels, rank, strong
    ((3, 3), 2, 1, True),
    ((33, 37), 3, 7, True),
    ((65, 34), 3, 17, True),
    ((64, 64), 4, 8, True),          # 64 atoms: 16 waves each
    ((50, 41), 3, 16, False),        # boxes of 1,000 rows: a workgroup per projection
    ((27, 25, 26), 3, 20, True),     # 320 atoms: 16 waves each
    ((224, 224), 5, 3, True),        # 1,024 atoms: 4 waves each
]


def build(case, prec):
    sizes, levels, r, strong = case
    n = int(np.prod(sizes))
    rng = np.random.default_rng(n + r)
    dt = np.float64 if prec == "f64" else np.float32
    cut = lambda a: a.astype(dt).astype(np.float64)
    U, V, X, Y = (cut(rng.standard_normal((n, c))) for c in (r, r, 8, 8))
    cls = dmhm_amd.HMat2d if len(sizes) == 2 else dmhm_amd.HMat3d
    H = cls.from_lowrank(sizes, levels, max(r, 4), strong, U, V,
                         precision=dmhm_amd.DMHM_F64 if prec == "f64" else dmhm_amd.DMHM_F32)
    return H, U, V, X, Y, dt


def check(got, L, R, X, Y, dt):
    n, r = L.shape
    ref = 0.5 * (L @ (R.T @ X)) - 2.0 * Y
    # Standard bound of nested sums (n + r + 4 roundings).
    bound = (n + r + 4) * np.finfo(dt).eps * (0.5 * np.abs(L) @ (np.abs(R).T @ np.abs(X)) + 2.0 * np.abs(Y))
    assert np.all(np.abs(got - ref) <= bound), float((np.abs(got - ref) / bound).max())


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_streaming_products(case, prec):
    H, U, V, X, Y, dt = build(case, prec)
    for k in (1, 2, 3, 5, 8):
        x, y = X[:, :k].astype(dt), Y[:, :k].astype(dt)
        check(H.Multiply(0.5, x, -2.0, y.copy(order="F")), U, V, X[:, :k], Y[:, :k], dt)
        check(H.TransposeMultiply(0.5, x, -2.0, y.copy(order="F")), V, U, X[:, :k], Y[:, :k], dt)


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_misaligned_strided_device_operands(prec):
    H, U, V, X, Y, dt = build(CASES[1], prec)
    n, k = X.shape[0], 3
    for op, L, R in (("N", U, V), ("T", V, U)):
        bufs = []
        for src in (X, Y):
            buf = torch.zeros((k, n + 5), dtype=torch.float64 if prec == "f64" else torch.float32, device="cuda")
            view = buf[:, 1:n + 1].t()          # starts one element in, leading dimension n + 5
            view.copy_(torch.from_numpy(src[:, :k].astype(dt)))
            bufs.append((buf, view))
        (_, x), (ybuf, y) = bufs
        (H.Multiply if op == "N" else H.TransposeMultiply)(0.5, x, -2.0, y)
        check(y.cpu().numpy(), L, R, X[:, :k], Y[:, :k], dt)
        assert float(ybuf[:, 0].abs().max()) == 0 and float(ybuf[:, n + 1:].abs().max()) == 0
