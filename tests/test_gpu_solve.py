"""The LU panels and thin solves (hbem_dense.hip, hbem_solve.hip) where their forms
change: blocks of 64 rows, panels of 32 columns held in registers up to 512, 1024,
2048 and 4096 rows, solve panels of 512 rows, one to eight right-hand sides.

sigma and dsigma of the randomized SVD against the oracle with the same test
matrix.  T = P (3 I + G / sqrt(n)) with a random row permutation P (every
pivot moves) is well conditioned (cond < 10): LU with partial pivoting errs by at
most ~10 n eps, q power iterations of two solves each by ten times that, so the
tolerance is 100 n eps.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def matrix(n, seed):
    rng = np.random.default_rng(seed)
    G = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(2 * n)
    return np.asfortranarray((3 * np.eye(n) + G)[rng.permutation(n)]), np.asfortranarray(G.T.copy())


def close(got, want, n):
    return np.all(np.abs(np.asarray(got) - np.asarray(want)) <= 100 * n * 2.0 ** -52 * max(1.0, np.abs(want).max()))


@pytest.mark.parametrize("n", [1, 2, 31, 33, 63, 64, 65, 127, 129, 511, 512, 513, 576, 577])
@pytest.mark.parametrize("nc", [1, 2, 3, 4, 5, 8])
def test_sizes(n, nc, H, O):
    if nc > n:
        pytest.skip("more right-hand sides than rows")
    T, Td = matrix(n, n)
    R = H.gaussian_test_matrix(n, nc, 7)
    assert close(H.randomized_svd.sv_der(T, Td, R, 2), O.sv_der(T, Td, R, 2), n)


@pytest.mark.parametrize("n", [1023, 1025, 1537])
@pytest.mark.parametrize("nc", [2, 3, 6])
def test_large_sizes(n, nc, H, O):
    T, _ = matrix(n, n)
    R = H.gaussian_test_matrix(n, nc, 7)
    assert close(H.randomized_svd.sv(T, R, 1), O.sv(T, R, 1), n)


def test_ties_take_the_first_row(H, O):
    """Entries of equal modulus in every column: the oracle's pivots (the first
    index), hence its sigma to rounding."""
    n = 96
    rng = np.random.default_rng(3)
    T = np.asfortranarray(rng.choice([1, -1, 1j, -1j], size=(n, n)) + 8.0 * np.eye(n)[rng.permutation(n)])
    R = H.gaussian_test_matrix(n, 2, 1)
    assert close(H.randomized_svd.sv(T, R, 2), O.sv(T, R, 2), n)


def test_singular_and_nan_columns_end(H):
    """A zero column and a column of NaNs: no hang, no finite sigma made up."""
    n = 200
    T, _ = matrix(n, 5)
    R = H.gaussian_test_matrix(n, 2, 1)
    T[:, 40] = 0.0
    assert not H.randomized_svd.sv(T, R, 2) > 1e-12
    T[:, 40] = np.nan
    assert np.isnan(H.randomized_svd.sv(T, R, 2))
