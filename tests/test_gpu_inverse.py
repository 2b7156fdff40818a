"""Gauss-Jordan inverse of matrices with NaN: where a column's remaining rows hold nothing but NaN
the pivot stays on the diagonal, so no index leaves the matrix (n = 1024 also fills the kernel's
LDS arrays); the result shows the NaN and the next inverse is unaffected."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [2, 4, 5, 16])
def test_inverse_of_nan(L):
    import dqmc_amd
    dqmc_amd.load()
    n = 4 * L * L
    print("inverse with NaN, n=%d" % n, flush=True)
    rng = np.random.default_rng(L)
    A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)) + 3.0 * np.eye(n)
    c = dqmc_amd.DQMC(dqmc_amd.Params(L=L, slices=20, hoppings=(1.0, 0.5, 0.5, 1.0), lam=1.0, r=1.0))
    want, ld = c.inv(A)
    for rows, cols in (([n // 2], [n // 3]), (range(n), [0]), (range(n), [n - 1]), (range(n), range(n))):
        B = A.copy()
        B[np.ix_(list(rows), list(cols))] = np.nan
        X, l = c.inv(B)
        assert np.isnan(X).any() and np.isnan(l)
        if len(cols) == n:
            assert np.isnan(X).all()
        X, l = c.inv(A)
        assert np.array_equal(X, want) and l == ld
    c.close()
