"""QR panels and dense leaf inverses at the edges of their kernels' tiles,
against exact products in float64. RoundedUpdate of factors whose last column
repeats the first has rank k - 1, so truncation to k - 1 reproduces the sum:
its error and the orthogonality of U are those of two Householder QRs and an
SVD of order k, a few k eps (50 k eps allowed)."""
import numpy as np
import pytest

import dmhm_amd
from dmhm_amd import workloads as W

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module", autouse=True)
def _init():
    dmhm_amd.init(0)
    yield


# Class edges in m (64, 256, 512, 1024 rows) and in k (groups of 4 and 8
# columns, the 24- and 40-column variants), and panels wider than tall.
@pytest.mark.parametrize("m,n,k", [(64, 63, 4), (65, 64, 5), (33, 15, 8), (17, 64, 9), (63, 62, 16), (64, 64, 17),
                                   (24, 64, 24), (20, 64, 24), (64, 3, 23), (64, 41, 25), (40, 64, 40), (30, 64, 37),
                                   (256, 255, 20), (257, 256, 24), (512, 300, 33), (513, 511, 24), (1024, 1, 12)])
@pytest.mark.parametrize("graded", [False, True])
def test_rounded_update_at_panel_edges(m, n, k, graded):
    print("case", m, n, k, graded, flush=True)
    rng = np.random.default_rng(1000 * m + 10 * n + k)
    U0, V0 = rng.standard_normal((m, k)), rng.standard_normal((n, k))
    U0[:, -1] = U0[:, 0]
    if graded:
        U0 *= np.logspace(0, -9, k)
        U0[:, -1] = U0[:, 0]
        U0[:, k // 2] = 0.0
    ka = k // 2
    want = U0[:, :ka] @ V0[:, :ka].T + 0.5 * U0[:, ka:] @ V0[:, ka:].T
    U, V = dmhm_amd.RoundedUpdate(k - 1, 1.0, (U0[:, :ka], V0[:, :ka]), 0.5, (U0[:, ka:], V0[:, ka:]))
    r = min(k - 1, m, n)
    assert U.shape == (m, r) and V.shape == (n, r)
    tol = 50 * k * EPS
    assert np.linalg.norm(U @ V.T - want) <= tol * np.linalg.norm(U0) * np.linalg.norm(V0)


# Panels of 4 columns (of 8 beyond 64 rows): one short, whole, one over, and
# the first and last size of each kernel.
@pytest.mark.parametrize("m", [1, 3, 4, 5, 31, 60, 61, 63, 64, 65, 72, 127, 128, 129, 255, 256, 257])
def test_leaf_inverse_at_panel_edges(m):
    print("case", m, flush=True)
    rng = np.random.default_rng(m)
    D = rng.standard_normal((m, m))
    D[np.diag_indices(m)] = 0.0 if m > 1 else 2.0            # every first pivot off the diagonal
    rowptr = np.arange(0, m * m + 1, m, dtype=np.int32)
    colind = np.tile(np.arange(m, dtype=np.int32), m)
    A = dmhm_amd.HMat2d.from_csr([m, 1], 1, 4, True, rowptr, colind, D.ravel().copy())
    X = A.DirectInvert().to_dense()
    # Gauss-Jordan with partial pivoting: forward error of a few m eps cond.
    want = np.linalg.inv(D)
    assert np.linalg.norm(X - want) <= 50 * m * EPS * np.linalg.cond(D) * np.linalg.norm(want)
