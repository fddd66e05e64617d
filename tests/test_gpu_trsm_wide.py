"""The triangular solve with many right-hand sides at the sizes where it can go
wrong: edges of the 16-column blocks, the 128-blocks and the groups of four,
ragged ends in both directions, and right-hand-side counts around a wave's 16
rows.  Integer solutions of integer systems must come out exactly."""
import ctypes as C

import numpy as np
import pytest

import libflame_amd as fla
from tests.cases import exact_tri
from tests.gpu_util import gpu_trsm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    fla.FLA_Init()
    yield


@pytest.mark.parametrize("n,nrhs", [(1, 33), (15, 64), (17, 40), (127, 33), (129, 65), (143, 100),
                                    (512, 49), (513, 40), (700, 37)])
@pytest.mark.parametrize("left", [True, False])
@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("trans", [True, False])
def test_exact(n, nrhs, left, lower, trans):
    unit = bool((n + nrhs) & 1)
    T = exact_tri(n, seed=n, lower=lower, unit=unit)
    # sparse off-diagonal part: the exact solutions stay small
    T = np.where(np.eye(n, dtype=bool) | (np.random.default_rng(n).random((n, n)) < 0.05), T, 0.0)
    X = np.random.default_rng(nrhs).integers(-4, 5, size=(n, nrhs) if left else (nrhs, n))
    op = T.T if trans else T
    B = op @ X if left else X @ op
    S = T.copy()
    if unit:
        np.fill_diagonal(S, 7.0)  # a unit diagonal is not read
    out = gpu_trsm(fla.FLA_LEFT if left else fla.FLA_RIGHT,
                   fla.FLA_LOWER_TRIANGULAR if lower else fla.FLA_UPPER_TRIANGULAR,
                   fla.FLA_TRANSPOSE if trans else fla.FLA_NO_TRANSPOSE,
                   fla.FLA_UNIT_DIAG if unit else fla.FLA_NONUNIT_DIAG, S, B.astype(np.float64))
    assert np.array_equal(out, X)


def _reference(T, B, left, lower, trans, unit):
    """dtrsm_'s substitution, one component at a time."""
    op = T.T if trans else T
    M, X = (op, B.copy()) if left else (op.T, B.T.copy())  # M X = B
    n = M.shape[0]
    fwd = lower != trans if left else lower == trans
    with np.errstate(divide="ignore", invalid="ignore"):
        for j in range(n) if fwd else range(n - 1, -1, -1):
            if not unit:
                X[j] /= M[j, j]
            rest = slice(j + 1, n) if fwd else slice(0, j)
            X[rest] -= np.outer(M[rest, j], X[j])
    return X if left else X.T


def _solve(T, B, left, lower, trans, unit=False):
    return gpu_trsm(fla.FLA_LEFT if left else fla.FLA_RIGHT,
                    fla.FLA_LOWER_TRIANGULAR if lower else fla.FLA_UPPER_TRIANGULAR,
                    fla.FLA_TRANSPOSE if trans else fla.FLA_NO_TRANSPOSE,
                    fla.FLA_UNIT_DIAG if unit else fla.FLA_NONUNIT_DIAG, T, B)


def _sparse_tri(n, lower):
    T = exact_tri(n, seed=n, lower=lower)
    return np.where(np.eye(n, dtype=bool) | (np.random.default_rng(n).random((n, n)) < 0.05), T, 0.0)


@pytest.mark.parametrize("at", [3, 9, 137])
@pytest.mark.parametrize("what", ["diagonal", "rhs"])
@pytest.mark.parametrize("left", [True, False])
@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("trans", [True, False])
def test_components_before_an_infinity_stay(at, what, left, lower, trans):
    """A zero on the diagonal or an infinite right-hand side at the at-th
    component solved changes that one and the later ones only."""
    n, nrhs = 200, 40
    T = _sparse_tri(n, lower)
    fwd = lower != trans if left else lower == trans
    j = at if fwd else n - 1 - at
    B = np.random.default_rng(at).integers(1, 5, size=(n, nrhs) if left else (nrhs, n)).astype(float)
    if what == "diagonal":
        T[j, j] = 0.0
    elif left:
        B[j, :] = np.inf
    else:
        B[:, j] = np.inf
    ref = _reference(T, B, left, lower, trans, False)
    out = _solve(T, B, left, lower, trans)
    done = [k if fwd else n - 1 - k for k in range(at)]
    ahead = ref[done] if left else ref[:, done]
    assert np.all(np.isfinite(ahead))
    assert np.array_equal(out[done] if left else out[:, done], ahead)
    assert np.array_equal(np.isfinite(out), np.isfinite(ref))


@pytest.mark.parametrize("lower", [True, False])
@pytest.mark.parametrize("trans", [True, False])
def test_left_solves_divide(lower, trans):
    """Exact quotients of a solve from the left come out exactly whatever the
    diagonal: by odd integers (49 (1/49) is not 1), by subnormal numbers
    (their reciprocals overflow) and by those whose reciprocals are subnormal."""
    n, nrhs = 150, 40
    rng = np.random.default_rng(n)
    T = _sparse_tri(n, lower)
    np.fill_diagonal(T, rng.choice([3.0, 49.0, 98.0, 103.0, -107.0], size=n))
    X = rng.integers(-4, 5, size=(n, nrhs)).astype(np.float64)
    out = _solve(T, (T.T if trans else T) @ X, True, lower, trans)
    assert np.array_equal(out, X)
    d = rng.choice([3 * 2.0**-1040, -7 * 2.0**-1060, 1.75 * 2.0**1023, 49.0], size=n)
    X = np.where(abs(d) < 1e-300, 2.0**40, 0.25)[:, None] * rng.integers(1, 4, size=(n, nrhs))
    B = d[:, None] * X
    assert np.array_equal(B / d[:, None], X) and np.all(np.isfinite(B))
    out = _solve(np.diag(d), B, True, lower, trans)
    assert np.array_equal(out, X)


def test_wide_solve_allocates_nothing():
    """A solve with many right-hand sides takes its block workspace from the
    library's start, at any order: the free device memory does not change, so
    the first call of a size can be captured."""
    hip = C.CDLL("libamdhip64.so")

    def free():
        f, t = C.c_size_t(0), C.c_size_t(0)
        assert hip.hipDeviceSynchronize() == 0
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    n, nrhs = 40000, 33
    dT, dB = fla.DeviceMatrix(n, n), fla.DeviceMatrix(n, nrhs)
    before = free()
    fla.check(fla.lib().fla_hip_dtrsm(fla.FLA_LEFT, fla.FLA_LOWER_TRIANGULAR, fla.FLA_NO_TRANSPOSE,
                                      fla.FLA_UNIT_DIAG, n, nrhs, 1.0, dT.ptr, dT.ld, dB.ptr,
                                      dB.ld))
    assert free() == before


@pytest.mark.parametrize("left,lower,trans", [(True, True, False), (True, True, True),
                                              (False, True, False), (False, False, False)])
def test_more_blocks_than_the_workspace_holds(left, lower, trans):
    """Past 64 diagonal blocks the workspace is written again, in both directions."""
    n, nrhs = 8192 + 700, 40
    rng = np.random.default_rng(8)
    T = np.zeros((n, n), order="F")
    i, j = rng.integers(0, n, size=(2, 6 * n))
    T[np.maximum(i, j), np.minimum(i, j)] = rng.integers(-2, 3, size=6 * n)
    if not lower:
        T = np.asfortranarray(T.T)
    np.fill_diagonal(T, rng.choice([1.0, -2.0, 4.0], size=n))
    X = rng.integers(-3, 4, size=(n, nrhs) if left else (nrhs, n)).astype(np.float64)
    op = T.T if trans else T
    out = _solve(T, op @ X if left else X @ op, left, lower, trans)
    assert np.array_equal(out, X)


def test_captured_call_replays():
    """A solve captured on the caller's stream gives the eager result on every
    replay, with the program's own copies and synchronisations in between."""
    hip, L = C.CDLL("libamdhip64.so"), fla.lib()
    n, nrhs = 700, 96
    T = _sparse_tri(n, True)
    B = np.asfortranarray(T @ np.random.default_rng(1).integers(-4, 5, size=(n, nrhs)))
    want = _solve(T, B, True, True, False)
    dT, dB = fla.DeviceMatrix.from_host(T), fla.DeviceMatrix.from_host(B)
    s, g, x = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(s)) == 0
    fla.check(L.fla_hip_set_stream(s))
    try:
        assert hip.hipStreamBeginCapture(s, 1) == 0  # thread local
        st = L.fla_hip_dtrsm(fla.FLA_LEFT, fla.FLA_LOWER_TRIANGULAR, fla.FLA_NO_TRANSPOSE,
                             fla.FLA_NONUNIT_DIAG, n, nrhs, 1.0, dT.ptr, dT.ld, dB.ptr, dB.ld)
        assert hip.hipStreamEndCapture(s, C.byref(g)) == 0
        fla.check(st)
    finally:
        fla.check(L.fla_hip_set_stream(None))
    assert np.array_equal(dB.download(), B)  # captured, not run
    assert hip.hipGraphInstantiate(C.byref(x), g, None, None, C.c_size_t(0)) == 0
    for _ in range(3):
        dB.upload(B)
        assert hip.hipGraphLaunch(x, s) == 0
        assert hip.hipStreamSynchronize(s) == 0
        assert np.array_equal(dB.download(), want)
        assert np.array_equal(_solve(T, B, True, True, False), want)
    assert hip.hipGraphExecDestroy(x) == 0 and hip.hipGraphDestroy(g) == 0
    assert hip.hipStreamDestroy(s) == 0
