"""The LDS-free 64 x 64 product kernel (few-tile shapes of C += A B'): tile,
wave and K-chunk edges, full and lower, exact on integers."""
import numpy as np
import pytest

import libflame_amd as fla
from tests.gpu_util import gpu_gemm, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    fla.FLA_Init()
    yield


@pytest.mark.parametrize("m,n", [(1, 1), (15, 33), (32, 64), (63, 65), (64, 64), (129, 31),
                                 (500, 130)])
@pytest.mark.parametrize("k", [1, 3, 4, 31, 32, 33, 64, 100, 128, 259])
def test_nt_product_exact(m, n, k):
    rng = np.random.default_rng(m + 7 * n + 31 * k)
    A, B, Cm = (rng.integers(-8, 9, size=s).astype(np.float64) for s in ((m, k), (n, k), (m, n)))
    out = gpu_gemm(fla.FLA_NO_TRANSPOSE, fla.FLA_TRANSPOSE, A, B, Cm, alpha=-2.0, beta=3.0)
    assert np.array_equal(out, -2.0 * (A @ B.T) + 3.0 * Cm)


@pytest.mark.parametrize("n", [1, 31, 64, 65, 200])
@pytest.mark.parametrize("k", [5, 128])
def test_lower_update_exact(n, k):
    rng = np.random.default_rng(n + 13 * k)
    A = rng.integers(-8, 9, size=(n, k)).astype(np.float64)
    Cm = rng.integers(-8, 9, size=(n, n)).astype(np.float64)
    dA, dC = to_dev(A), to_dev(Cm)
    fla.check(fla.lib().fla_hip_dsyrk(fla.FLA_LOWER_TRIANGULAR, fla.FLA_NO_TRANSPOSE, n, k, -1.0,
                                      dA.ptr, dA.ld, 1.0, dC.ptr, dC.ld))
    fla.synchronize()
    ref = np.where(np.tril(np.ones((n, n), bool)), Cm - A @ A.T, Cm)
    assert np.array_equal(dC.download(), ref)
