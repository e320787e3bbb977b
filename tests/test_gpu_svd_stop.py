"""The SVD's last sweep: Compress of triangular matrices whose rows are nearly
orthogonal, so that the QR leaves them as they are and every rotation of the
first sweep is small, and of random ones. V's columns are then the rotated
columns themselves. Their cosines stay at the 1e-15 below which the kernel
takes a pair as orthogonal, plus four roundings of the columns; singular
values are within k eps of numpy's relative to the largest."""
import numpy as np
import pytest

import dmhm_amd

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def cosines(V):
    V = V.astype(np.longdouble)
    V = V / np.sqrt((V * V).sum(axis=0))
    G = np.abs(V.T @ V)
    np.fill_diagonal(G, 0)
    return float(G.max())


@pytest.mark.parametrize("k", [24, 40, 64])
@pytest.mark.parametrize("cos", [1e-9, 3e-9, 4.5e-9, 6e-9])
def test_small_rotations_leave_orthogonal_columns(k, cos):
    R = np.triu(np.full((k, k), cos), 1) + np.eye(k)
    R *= 1.35 ** -np.arange(k)[:, None]
    U, V = dmhm_amd.Compress(k, R)
    assert V.shape == (k, k)
    assert cosines(V) <= 1e-15 + 4 * EPS / 2
    assert np.abs(np.linalg.norm(V, axis=0) - np.linalg.svd(R)[1]).max() <= k * EPS


@pytest.mark.parametrize("k", [7, 20, 24, 36, 40, 63, 64])
def test_random_factors(k):
    rng = np.random.default_rng(k)
    D = np.linalg.qr(rng.standard_normal((64, k)))[0] * rng.uniform(0.5, 1.0, k) @ rng.standard_normal((k, k))
    U, V = dmhm_amd.Compress(k, D)
    s = np.linalg.svd(D)[1]
    assert V.shape[1] == k and np.abs(np.linalg.norm(V, axis=0) - s).max() <= k * EPS * s[0]
    # Rounding of U V^T and of the QR: 10 k roundings.
    assert np.linalg.norm(U @ V.T - D) <= 10 * k * EPS * np.linalg.norm(D)
