"""The LU sub-panel kernel where it can go wrong: heights around the 512
threads and the 1024 rows of a workgroup, ragged last sub-panels, and NaN or
infinite entries in workgroups other than the pivot's."""
import ctypes as C

import numpy as np
import pytest

import libflame_amd as fla
from tests.cases import exact_lu
from tests.gpu_util import gpu_lu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    fla.FLA_Init()
    yield


@pytest.mark.parametrize("m,n", [(33, 33), (63, 40), (511, 70), (513, 33), (1023, 65), (1024, 32),
                                 (1025, 97), (2049, 160), (1100, 129)])
def test_sub_panel_exact(m, n):
    A, L, U, p = exact_lu(n, seed=m + n, m=m)
    out, pv, r = gpu_lu(A)
    assert r == fla.FLA_SUCCESS
    assert np.array_equal(pv, p)
    assert np.array_equal(np.tril(out[:, :n], -1), np.tril(L, -1))
    assert np.array_equal(np.triu(out[:n, :]), U)


@pytest.mark.parametrize("rows", [[7], [600], [1500], [40, 2100], [2199]])
def test_nan_restart_across_workgroups(orc, rows):
    A = np.asfortranarray(orc.gen_lu_c2(3, 2200, 40))
    for r in rows:
        A[r, 0] = np.nan
    _, pv, _ = gpu_lu(A)
    _, pref, _ = orc.lu_piv(A)
    assert pv[0] == pref[0]


@pytest.mark.parametrize("m", [100, 1500])
def test_infinite_row_keeps_finished_rows(orc, m):
    """An infinity right of the first columns reaches the rows below its pivot
    row only: finished rows of U and the columns left of it stay finite."""
    n, c = 32, 9
    A = np.asfortranarray(orc.gen_lu_c2(5, m, n))
    A[0, c] = np.inf
    out, pv, _ = gpu_lu(A)
    ref, pref, _ = orc.lu_piv(A)
    assert np.array_equal(pv[:c], pref[:c])
    assert np.array_equal(np.isfinite(out[:, :c]), np.isfinite(ref[:, :c]))
    k = next(i for i in range(n) if not np.isfinite(ref[i, c]))
    assert np.all(np.isfinite(out[:k, :]))


@pytest.mark.parametrize("m", [560, 600, 1500])
@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("c", [1, 9])
def test_non_finite_pivot_row_reaches_every_row(orc, m, value, c):
    """A pivot row holding an infinity or NaN updates every row below it, those
    of a thread's second register row (512 and up) too, and the pivots chosen
    from them follow (in the next column a finite row among NaNs would be
    chosen, or be scaled to zero by an infinite pivot)."""
    n = 32
    A = np.asfortranarray(orc.gen_lu_c2(5, m, n))
    A[0, 0] = 8.0  # the first pivot
    A[0, c] = value
    out, pv, _ = gpu_lu(A)
    ref, pref, _ = orc.lu_piv(A)
    assert np.array_equal(pv, pref)
    assert np.array_equal(np.isfinite(out), np.isfinite(ref))
    assert np.array_equal(np.isnan(out), np.isnan(ref))


def test_after_an_expired_wait_no_rows_move(orc):
    """Panels launched after a bounded wait of the factorization expired (here:
    its flag is set beforehand) do nothing, and the interchanges queued behind
    them move no rows, though the lists held a taller panel's before."""
    L = fla.lib()
    setup = L["_Z18fla_lu_panel_setupiPi"]
    run = L["_Z16fla_lu_panel_runP12ihipStream_tiiiPdliPiS2_"]
    gather = L["_Z18fla_lu_gather_rowsP12ihipStream_tiiPdl"]
    setup.argtypes = [C.c_int, C.c_void_p]
    run.argtypes = [C.c_void_p] + [C.c_int] * 3 + [C.c_void_p, C.c_long, C.c_int] + [C.c_void_p] * 2
    gather.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_long]
    hip = C.CDLL("libamdhip64.so")
    w, piv = 128, fla.DeviceMatrix(128, 1, np.int32)
    flags = fla.DeviceMatrix(2, 1, np.int32)  # expired, info

    def panel(A, expired):
        flags.upload(np.array([[expired], [-1]], dtype=np.int32))
        d = fla.DeviceMatrix.from_host(A)
        fla.check(setup(d.ld, flags.ptr))
        m = A.shape[0] - 40  # the last 40 rows stay outside
        fla.check(run(None, 0, m, w, d.ptr, d.ld, 0, piv.ptr, flags.ptr.value + 4))
        c = fla.DeviceMatrix.from_host(A)
        fla.check(gather(None, 0, w, c.ptr, c.ld))
        assert hip.hipDeviceSynchronize() == 0
        return d.download(), c.download()

    tall = np.asfortranarray(orc.gen_lu_c2(3, 3040, w))
    _, moved = panel(tall, 0)
    assert not np.array_equal(moved, tall)  # its lists move rows
    low = np.asfortranarray(orc.gen_lu_c2(4, 340, w))
    out, moved = panel(low, 1)
    assert np.array_equal(moved, low)
    assert np.array_equal(out[300:], low[300:])
    _, moved = panel(low, 0)
    assert not np.array_equal(moved, low) and np.array_equal(moved[300:], low[300:])
