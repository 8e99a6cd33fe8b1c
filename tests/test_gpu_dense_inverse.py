"""Inverse of a dense SPD matrix by the blocked Cholesky (phd_dense.hip) against numpy."""
import numpy as np
import pytest

from diffphd_amd import _lib

pytestmark = pytest.mark.gpu


def _inverse(A, precision):
    n = A.shape[0]
    a_arr, a_p = _lib.dptr(np.asarray(A, dtype=np.float64).ravel(order="F"))
    x_arr, x_p = _lib.dptr(np.zeros(n * n))
    rc = _lib.lib().phd_dense_spd_inverse(n, a_p, x_p, precision)
    return rc, x_arr.copy().reshape(n, n, order="F")


# One block and its padding (1, 63, 64), the first block row of Y below the matrix
# (65), and around the groups of four block columns whose trailing updates go
# together: 5, 8 and 9 blocks, and 13, which leaves a partial last group.
@pytest.mark.parametrize("n", [1, 63, 64, 65, 260, 512, 513, 800])
@pytest.mark.parametrize("precision,eps", [(0, 2.0**-53), (1, 2.0**-24)])
def test_dense_spd_inverse_matches_numpy(n, precision, eps):
    rng = np.random.default_rng(n)
    B = rng.standard_normal((n, n))
    A = B @ B.T + n * np.eye(n)
    rc, X = _inverse(A, precision)
    assert rc == 0
    assert np.array_equal(X, X.T)
    # Cholesky and the triangular inverse are backward stable: the error of an entry
    # is at most a small multiple of n eps cond(A) |A^-1|, cond(A) < 6 here
    err = np.linalg.norm(X - np.linalg.inv(A), 2)
    bound = 10 * n * eps * np.linalg.cond(A) * np.linalg.norm(np.linalg.inv(A), 2) + 1e-300
    print(n, precision, err, bound)
    assert err <= bound


@pytest.mark.parametrize("precision", [0, 1])
def test_dense_spd_inverse_reports_indefinite(precision):
    A = np.eye(330)
    A[200, 200] = -1.0
    assert _inverse(A, precision)[0] == 1
