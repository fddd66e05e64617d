"""The left-looking batched Cholesky and solve where it can go wrong: orders
around the 16-row blocks and the eight waves' turns, leading dimensions larger
than the order, right-hand-side counts around 16, and failing columns.  Exact
integer systems: factors and solutions must come out bit for bit."""
import ctypes as C

import numpy as np
import pytest

import libflame_amd as fla
from tests.cases import exact_spd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    fla.FLA_Init()
    yield


def _run(dtype, mats, rhs, pad):
    cnt = len(mats)
    dA, dB = [], []
    for a, b in zip(mats, rhs):
        n = a.shape[0]
        A = np.full((n + pad, n), 77.0, order="F")
        A[:n] = a
        B = np.full((n + pad, b.shape[1]), 55.0, order="F")
        B[:n] = b
        dA.append(fla.DeviceMatrix.from_host(A, dtype))
        dB.append(fla.DeviceMatrix.from_host(B, dtype))
    ptr = lambda v: (C.c_void_p * cnt)(*[x.ptr.value for x in v])  # noqa: E731
    ints = lambda v: (C.c_int * cnt)(*[int(x) for x in v])  # noqa: E731
    info = fla.DeviceMatrix(cnt, 1, np.int32)
    L = fla.lib()
    f = L.fla_hip_dposv_batched if dtype == np.float64 else L.fla_hip_sposv_batched
    fla.check(f(C.c_int(cnt), ints([a.shape[0] for a in mats]), ptr(dA), ints([d.ld for d in dA]),
                ptr(dB), ints([d.ld for d in dB]), ints([b.shape[1] for b in rhs]), info.ptr))
    fla.synchronize()
    return [d.download() for d in dA], [d.download() for d in dB], info.download().ravel()


def _spd(n, seed):
    """A sparse closed form, so that FP32 stays exact and solutions small."""
    _, F = exact_spd(n, seed)
    keep = np.random.default_rng(seed).random((n, n)) < 0.06
    F = np.where(keep | np.eye(n, dtype=bool), F, 0.0)
    return F @ F.T, F


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("pad", [0, 3])
def test_exact(dtype, pad):
    ns = [1, 15, 16, 17, 31, 33, 48, 49, 127, 128, 129, 143, 145, 257, 497, 511, 512]
    rs = [1, 2, 8, 15, 16, 17, 31, 33, 40]
    mats, facs, xs = [], [], []
    for i, n in enumerate(ns):
        A, F = _spd(n, n + 1)
        mats.append(A)
        facs.append(F)
        # only a few nonzeros: the triangular systems' intermediate values stay small
        X = np.zeros((n, rs[i % len(rs)]))
        X[:: max(1, n // 5)] = np.random.default_rng(n).integers(-2, 3, size=X[:: max(1, n // 5)].shape)
        xs.append(X)
    out, sol, info = _run(dtype, mats, [a @ x for a, x in zip(mats, xs)], pad)
    assert np.all(info == fla.FLA_SUCCESS)
    for n, A, F, X, o, s in zip(ns, mats, facs, xs, out, sol):
        assert np.array_equal(np.tril(o[:n]), F), n
        assert np.array_equal(np.triu(o[:n], 1), np.triu(A, 1)), n
        assert np.all(o[n:] == 77.0) and np.all(s[n:] == 55.0), n
        assert np.array_equal(s[:n], X), n


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_failing_column(dtype):
    cols = [0, 5, 15, 16, 31, 47, 100]
    mats = []
    for k in cols:
        A, F = _spd(101, 7)
        A[k, k] -= F[k, k] ** 2 + 1.0
        mats.append(A)
    _, _, info = _run(dtype, mats, [np.ones((101, 2))] * len(cols), 0)
    assert list(info) == cols


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_empty_matrices_and_negative_counts(dtype):
    """An item of order 0 touches nothing, whatever its matrix pointer and
    right-hand-side count; a negative count is no right-hand sides."""
    A, F = _spd(40, 7)
    X = np.full((40, 2), 3.0)
    ns, rs = [40, 0, 40, 0], [2, 5, -40, 1]
    dA = [fla.DeviceMatrix.from_host(np.asfortranarray(A), dtype) for _ in ns]
    dB = [fla.DeviceMatrix.from_host(np.asfortranarray(A @ X), dtype) for _ in ns]
    pA = (C.c_void_p * 4)(dA[0].ptr.value, None, dA[2].ptr.value, dA[3].ptr.value)
    pB = (C.c_void_p * 4)(*[b.ptr.value for b in dB])
    ints = lambda v: (C.c_int * 4)(*v)  # noqa: E731
    info = fla.DeviceMatrix(4, 1, np.int32)
    L = fla.lib()
    f = L.fla_hip_dposv_batched if dtype == np.float64 else L.fla_hip_sposv_batched
    fla.check(f(C.c_int(4), ints(ns), pA, ints([40] * 4), pB, ints([40] * 4), ints(rs), info.ptr))
    fla.synchronize()
    assert np.all(info.download() == fla.FLA_SUCCESS)
    assert np.array_equal(np.tril(dA[0].download()), F)
    assert np.array_equal(np.tril(dA[2].download()), F)
    assert np.array_equal(dA[3].download(), A)
    assert np.array_equal(dB[0].download(), X)
    for q in (1, 2, 3):
        assert np.array_equal(dB[q].download(), A @ X), q


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_entries_before_an_infinity_stay(dtype):
    """An infinity at (i, j) makes row i fail; what the row holds left of
    column j is the factor's, in the same 16 columns too."""
    at = [(40, 9), (40, 20), (95, 3), (99, 70)]
    A, F = _spd(101, 7)
    mats = []
    for i, j in at:
        M = A.copy()
        M[i, j] = np.inf
        mats.append(M)
    out, _, info = _run(dtype, mats, [np.ones((101, 2))] * len(at), 0)
    assert list(info) == [i for i, _ in at]
    for (i, j), o in zip(at, out):
        assert np.array_equal(o[i, :j], F[i, :j]), (i, j)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_solves_divide(dtype):
    """Exact quotients come out exactly (49 (1/49) is not 1), and infinities, NaN
    and overflowing quotients as a division gives them."""
    d = np.resize([3.0, 49.0, 98.0, 103.0, 107.0], 40)
    X = np.random.default_rng(3).integers(-4, 5, size=(40, 9)).astype(float)
    A = np.diag(d * d)
    big = 0.75 * float(np.finfo(dtype).max)
    special = np.array([[np.inf, -np.inf, np.nan, 0.0, big, -big]])
    out, sol, info = _run(dtype, [A, np.array([[0.25]])], [A @ X, special], 0)
    assert np.all(info == fla.FLA_SUCCESS)
    assert np.array_equal(out[0], np.diag(d))
    assert np.array_equal(sol[0], X)
    assert np.array_equal(sol[1], [[np.inf, -np.inf, np.nan, 0.0, np.inf, -np.inf]], equal_nan=True)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_failing_matrix_keeps_finished_columns(dtype):
    """The columns before the failing one are the factor's in every row, those
    of its own 16-column block too."""
    cols = [5, 15, 16, 21, 47, 100]
    A, F = _spd(101, 7)
    mats = []
    for k in cols:
        M = A.copy()
        M[k, k] -= F[k, k] ** 2 + 1.0
        mats.append(M)
    out, _, info = _run(dtype, mats, [np.ones((101, 2))] * len(cols), 0)
    assert list(info) == cols
    for k, o in zip(cols, out):
        assert np.array_equal(np.tril(o)[:, :k], F[:, :k]), k
