"""The dense fronts of the host factorization at the edges of their panels and lanes."""
import numpy as np
import pytest

from diffphd_amd import _lib


# A full matrix is one front. Panels have 48 columns and rows go eight at a time, two
# rows of the trailing update together: 7, 8, 9 and 47, 48, 49 stand around one of each,
# 57 leaves nine rows below a full panel, 97 a last panel of one column; 700 is past the
# size from which the panels are shared among threads.
@pytest.mark.parametrize("n", [1, 7, 8, 9, 47, 48, 49, 57, 97, 700])
def test_full_front_inverts(n):
    rng = np.random.default_rng(n)
    B = rng.standard_normal((n, n))
    A = B @ B.T / n + 2.0 * np.eye(n)
    app = _lib.iptr(np.arange(0, n * n + 1, n))
    aip = _lib.iptr(np.tile(np.arange(n), n))
    axp = _lib.dptr(A.ravel())
    xp = _lib.dptr(rng.uniform(0, 1, 3 * n))
    out, op = _lib.dptr(np.zeros(7))
    assert _lib.lib().phd_host_factor_check(n, app[1], aip[1], axp[1], xp[1], op) == 0
    # |S^T S A - I| <= a small multiple of n eps cond(A), cond(A) <= 3
    print(n, out[:3])
    assert out[0] <= 10 * n * 2.0**-53 * 3 + 1e-15
    assert out[6] == 0


def test_full_front_reports_indefinite():
    n = 60
    A = np.eye(n)
    A[53, 53] = -1.0
    A[A == 0] = 1e-9
    app = _lib.iptr(np.arange(0, n * n + 1, n))
    aip = _lib.iptr(np.tile(np.arange(n), n))
    axp = _lib.dptr(A.ravel())
    xp = _lib.dptr(np.random.default_rng(1).uniform(0, 1, 3 * n))
    out, op = _lib.dptr(np.zeros(7))
    assert _lib.lib().phd_host_factor_check(n, app[1], aip[1], axp[1], xp[1], op) != 0
