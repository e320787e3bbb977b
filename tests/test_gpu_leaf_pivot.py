"""The pivot of a dense leaf inverse of more than 64 rows is the column's
largest entry on all 53 bits. Two candidates x < y agree in their first 20
bits; x / y = 1 - 2^-23, and 1 / y is a double to 1e-7 of its rounding, so the
elimination with pivot y is exact and one row of the inverse comes out exactly.
With pivot x, y / x has no finite expansion and that row is off by 64 ulps."""
import numpy as np
import pytest

import dmhm_amd

pytestmark = pytest.mark.gpu

Y = 889702353 / 2.0 ** 29
X = Y * (1 - 2.0 ** -23)


def test_the_two_candidates():
    y, x = np.array([Y]).view(np.uint64)[0], np.array([X]).view(np.uint64)[0]
    assert x < y and x >> np.uint64(32) == y >> np.uint64(32)
    assert X == Y - Y * 2.0 ** -23 and X * (1 / Y) == 1 - 2.0 ** -23


@pytest.mark.parametrize("m", [65, 128, 129, 200, 256])
@pytest.mark.parametrize("sign", [1, -1])
def test_largest_entry_is_the_pivot(m, sign):
    for r1, r2 in ((2, 7), (5, m - 3)):
        D = np.eye(m)
        D[r1, r1], D[r1, r2], D[r2, r1], D[r2, r2] = X, 1.0, sign * Y, sign
        rowptr = np.arange(0, m * m + 1, m, dtype=np.int32)
        colind = np.tile(np.arange(m, dtype=np.int32), m)
        A = dmhm_amd.HMat2d.from_csr([m, 1], 1, 4, True, rowptr, colind, D.ravel().copy())
        got = A.DirectInvert().to_dense()
        assert got[r2, r1] == 2.0 ** 23 and got[r2, r2] == -sign * (2.0 ** 23 - 1)
