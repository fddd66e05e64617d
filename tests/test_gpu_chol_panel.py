"""The register-resident diagonal factor and the panel solve of FLA_Chol at the
sizes and scales where they can go wrong: 16-column block edges inside the
last 128-block, row counts around a wave's 16 rows, and pivots whose root and
reciprocal leave the fast iteration's range.  Exact closed forms: every
factor must come out bit for bit."""
import numpy as np
import pytest

import libflame_amd as fla
from tests.cases import exact_spd
from tests.gpu_util import gpu_chol

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    fla.FLA_Init()
    yield


@pytest.mark.parametrize("n", [15, 16, 17, 33, 112, 113, 143, 144, 145, 191, 193, 400])
def test_panel_block_edges_exact(n):
    A, F = exact_spd(n, seed=3 * n + 1)
    out, r = gpu_chol(A)
    assert r == fla.FLA_SUCCESS
    assert np.array_equal(np.tril(out), F)
    assert np.array_equal(np.triu(out, 1), np.triu(A, 1))


@pytest.mark.parametrize("e", [-400, -348, 420, 500])
@pytest.mark.parametrize("n", [20, 150])
def test_scaled_pivots_exact(n, e):
    """A 2^(2e): L is the closed form times 2^e (pivots below 2^-700 and above
    2^1000 take the library root and division)."""
    A, F = exact_spd(n, seed=n)
    with np.errstate(over="ignore"):
        S = np.ldexp(A, 2 * e)
    if not np.all(np.isfinite(S)):
        pytest.skip("the scaled matrix overflows")
    out, r = gpu_chol(S)
    assert r == fla.FLA_SUCCESS
    assert np.array_equal(np.tril(out), np.ldexp(F, e))


@pytest.mark.parametrize("n,i,j", [(100, 40, 9), (100, 40, 20), (300, 250, 5), (300, 250, 137)])
def test_entries_before_an_infinity_stay(n, i, j):
    """An infinity at (i, j) makes row i fail; what the row holds left of
    column j is the factor's, in the same 16 columns too."""
    A, F = exact_spd(n, seed=n)
    A[i, j] = np.inf
    out, r = gpu_chol(A)
    assert r == i
    assert np.array_equal(out[i, :j], F[i, :j])


@pytest.mark.parametrize("n", [100, 128])
def test_sums_of_sixteen_terms(n):
    """The diagonal factor sums sixteen terms from zero before it subtracts
    them.  A model of its operations in that order is 0.9e-16 to 1.1e-16 off
    a wider-precision factor of these matrices, one that subtracts term by term
    1.7e-16 to 2.3e-16."""
    for seed in range(4):
        B = np.random.default_rng(seed).standard_normal((n, n))
        A = B @ B.T / n + np.eye(n)
        A = np.asfortranarray((A + A.T) / 2)
        R = A.astype(np.longdouble)
        for j in range(n):
            R[j, j] = np.sqrt(R[j, j])
            R[j + 1:, j] /= R[j, j]
            R[j + 1:, j + 1:] -= np.outer(R[j + 1:, j], R[j + 1:, j])
        R = np.tril(R)
        out, r = gpu_chol(A)
        assert r == fla.FLA_SUCCESS
        err = np.linalg.norm((np.tril(out) - R).astype(float)) / np.linalg.norm(R.astype(float))
        assert err < 1.4e-16, (seed, err)


@pytest.mark.parametrize("k", [5, 16, 40, 63, 95, 111, 127, 135])
def test_failing_column_keeps_finished_blocks(k):
    """Column k's pivot fails: the 16-column blocks before it are the factor's
    in all rows of the diagonal block."""
    n = 200
    A, F = exact_spd(n, seed=11)
    A[k, k] -= F[k, k] ** 2 + 1.0
    out, r = gpu_chol(A)
    assert r == k
    rows, cols = 128 * (k // 128) + 128, k // 16 * 16
    assert np.array_equal(np.tril(out)[:rows, :cols], F[:rows, :cols])
