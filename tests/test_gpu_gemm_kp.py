"""The LDS product kernel in every layout where its edge handling differs: last
rows and columns, K remainders, odd leading dimensions (16-byte loads at 8-byte
alignment) and more tiles than CUs; exact on integers."""
import numpy as np
import pytest

import libflame_amd as fla
from tests.gpu_util import gpu_gemm

pytestmark = pytest.mark.gpu
N, T = fla.FLA_NO_TRANSPOSE, fla.FLA_TRANSPOSE


@pytest.fixture(scope="module", autouse=True)
def _init():
    fla.FLA_Init()
    yield


@pytest.mark.parametrize("ta,tb", [(N, N), (N, T), (T, N), (T, T)])
@pytest.mark.parametrize("m,n,k", [(129, 127, 15), (255, 1, 33), (1, 200, 47), (384, 256, 32),
                                   (2101, 2175, 21), (2176, 2176, 16)])
def test_layouts_exact(ta, tb, m, n, k):
    rng = np.random.default_rng(m + n + k)
    A = rng.integers(-8, 9, size=(m, k) if ta == N else (k, m)).astype(np.float64)
    B = rng.integers(-8, 9, size=(k, n) if tb == N else (n, k)).astype(np.float64)
    Cm = rng.integers(-8, 9, size=(m, n)).astype(np.float64)
    out = gpu_gemm(ta, tb, A, B, Cm, alpha=-1.0, beta=2.0)
    ref = 2.0 * Cm - (A if ta == N else A.T) @ (B if tb == N else B.T)
    assert np.array_equal(out, ref)
