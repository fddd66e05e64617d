"""Performance cases: the factorizations and solves that programs have this library do.

Every case is one pass through the public entry points (FLA_Chol, FLA_LU_piv, the
solves on their factors, the mixed-precision solve, the batched calls and the
Cholesky adjoint) on matrices that are already in device memory.  A call that
factors in place gets a fresh copy of its matrix in the same pass, as a program
does that still needs the matrix (residuals, refinement).

A case's "kind" is one of

  chol        FLA_Chol of one SPD matrix
  spd_solve   FLA_Chol and FLA_Chol_solve: one system, a few right-hand sides
  lu          FLA_LU_piv of one general matrix
  lu_solve    FLA_LU_piv and FLA_LU_piv_solve
  chol_solve  FLA_Chol_solve with a factor that the program keeps
  posv_batch  fla_hip_{d,s}posv_batched: uneven SPD systems in one call
  gesv_batch  fla_hip_dgesv_batched: uneven general systems in one call
  mixed       fla_hip_dsposv: reduced-precision factor, refined to FP64
  adjoint     FLA_Chol_adjoint: reverse mode of the factorization
"""
import ctypes as C
import math
import random

import torch

import libflame_amd as fla

LOWER, UPPER = fla.FLA_LOWER_TRIANGULAR, fla.FLA_UPPER_TRIANGULAR
UPLO = {"lower": LOWER, "upper": UPPER}
DEV = "cuda"


def listed():
    return [
        # The smallest calls: one small covariance or normal-equations matrix,
        # where the launches and the host path are the time.
        {"name": "chol_n100", "kind": "chol", "n": 100, "uplo": "lower"},
        # The ordinary small matrix (the configuration of the parity tests).
        {"name": "chol_n1024", "kind": "chol", "n": 1024, "uplo": "lower"},
        # One odd-sized system solved from scratch, upper triangle stored.
        {"name": "spd_solve_n5003", "kind": "spd_solve", "n": 5003, "nrhs": 7, "uplo": "upper"},
        # The largest factorization: the benchmark's headline workload.
        {"name": "chol_n32768", "kind": "chol", "n": 32768, "uplo": "lower"},
        # A small odd general system.
        {"name": "lu_solve_n1531", "kind": "lu_solve", "n": 1531, "nrhs": 3},
        # The large LU of the benchmark (well-separated pivots).
        {"name": "lu_n16384", "kind": "lu", "m": 16384, "n": 16384},
        # Many solves with one kept factor: one call of them, 16 right-hand sides.
        {"name": "chol_solve_n16384", "kind": "chol_solve", "n": 16384, "nrhs": 16,
         "uplo": "lower"},
        # Thousands of small uneven systems in one call, FP64 and FP32.
        {"name": "dposv_batch_4096", "kind": "posv_batch", "dtype": "f64", "count": 4096,
         "nmin": 32, "nmax": 512, "sizes": 1},
        {"name": "sposv_batch_4096", "kind": "posv_batch", "dtype": "f32", "count": 4096,
         "nmin": 32, "nmax": 512, "sizes": 2},
        # The same for general matrices.
        {"name": "dgesv_batch_4096", "kind": "gesv_batch", "count": 4096, "nmin": 32,
         "nmax": 512, "sizes": 3},
        # A large system solved to FP64 accuracy from an FP32 factorization.
        {"name": "mixed_n16384", "kind": "mixed", "n": 16384, "nrhs": 8, "kappa": 100.0},
        # The backward direction: the gradient through one factorization (the
        # order of the Gaussian-process benchmark).
        {"name": "adjoint_n8192", "kind": "adjoint", "n": 8192},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["chol", "chol", "spd_solve", "lu", "lu_solve", "chol_solve", "posv_batch",
                       "posv_batch", "gesv_batch", "mixed", "adjoint"])
    c = {"kind": kind}
    if kind == "chol":
        c.update(n=_log_int(rng, 48, 24000), uplo=rng.choice(["lower", "upper"]))
    elif kind == "spd_solve":
        c.update(n=_log_int(rng, 150, 12000), nrhs=_log_int(rng, 1, 40),
                 uplo=rng.choice(["lower", "upper"]))
    elif kind == "lu":
        m = _log_int(rng, 200, 14000)
        c.update(m=m, n=m if rng.random() < 0.5 else max(64, int(m * rng.uniform(0.3, 1.0))))
    elif kind == "lu_solve":
        c.update(n=_log_int(rng, 100, 6000), nrhs=_log_int(rng, 1, 20))
    elif kind == "chol_solve":
        c.update(n=_log_int(rng, 500, 20000), nrhs=_log_int(rng, 1, 32),
                 uplo=rng.choice(["lower", "upper"]))
    elif kind in ("posv_batch", "gesv_batch"):
        if kind == "posv_batch":
            c["dtype"] = rng.choice(["f64", "f32"])
        lo = _log_int(rng, 8, 128)
        c.update(count=_log_int(rng, 200, 4096), nmin=lo, nmax=rng.randint(lo, 512),
                 sizes=rng.randint(1, 10 ** 6))
    elif kind == "mixed":
        c.update(n=_log_int(rng, 2000, 14000), nrhs=rng.randint(1, 16),
                 kappa=rng.choice([1e2, 1e4]))
    else:
        c.update(n=_log_int(rng, 400, 8192))
    return c


# ---- inputs ------------------------------------------------------------------
# A column-major m x n matrix is held as a contiguous torch tensor t of shape
# (n, m): t[j, i] is entry (i, j).

class Matrix:
    """A torch tensor as the library's column-major m x n device matrix."""

    def __init__(self, t):
        self.t, self.n, self.m = t, t.shape[0], t.shape[1]
        self.ld = self.m
        self.ptr = C.c_void_p(t.data_ptr())

    def obj(self):
        dt = fla.FLA_INT if self.t.dtype == torch.int32 else fla.FLA_DOUBLE
        return fla.Obj.attach(self.t.data_ptr(), self.m, self.n, dt, self.ld)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _spd(n, g):
    """B B'/n + I, B i.i.d. N(0,1) (full symmetric storage)."""
    B = torch.randn(n, n, dtype=torch.float64, device=DEV, generator=g)
    A = B @ B.T
    del B
    A.div_(n)
    A.diagonal().add_(1.0)
    return A


def _normal(shape, g, dtype=torch.float64):
    return torch.randn(shape, dtype=dtype, device=DEV, generator=g)


def _general(m, n, g):
    """U[-1,1] entries, row i scaled by 10^(-i/max(m,n)): well-separated pivots."""
    t = torch.rand(n, m, dtype=torch.float64, device=DEV, generator=g).mul_(2).sub_(1)
    rows = torch.arange(m, dtype=torch.float64, device=DEV)
    return t.mul_(torch.pow(10.0, -rows / max(m, n)))


def _spd_kappa(n, kappa, g):
    """Q diag(s) Q', s log-spaced on [1, kappa], Q a product of 64 reflectors."""
    s = torch.logspace(0, math.log10(kappa), n, dtype=torch.float64, device=DEV)
    A = torch.diag(s)
    for _ in range(64):
        v = _normal((n,), g)
        v /= v.norm()
        w = A @ v
        u = 2.0 * w - 2.0 * torch.dot(v, w) * v
        A.addr_(u, v, alpha=-1.0)
        A.addr_(v, u, alpha=-1.0)
    return A


def _tri(A, uplo):
    """The stored triangle of a symmetric matrix, zeros elsewhere (in our layout
    entry (i, j) with i >= j is t[j, i]: the tensor's upper triangle)."""
    return torch.triu(A) if uplo == "lower" else torch.tril(A)


def _batch_shape(case):
    r = random.Random(case["sizes"])
    ns = [r.randint(case["nmin"], case["nmax"]) for _ in range(case["count"])]
    return ns, [r.randint(1, 8) for _ in ns]


def _offsets(sizes):
    off = [0]
    for s in sizes:
        off.append(off[-1] + s)
    return off


def _batch_values(case, seed):
    """The matrices and right-hand sides, back to back in two flat tensors."""
    ns, rs = _batch_shape(case)
    oa, ob = _offsets([n * n for n in ns]), _offsets([n * r for n, r in zip(ns, rs)])
    g = _gen(seed)
    dt = torch.float32 if case.get("dtype") == "f32" else torch.float64
    B = _normal((ob[-1],), g, dt)
    if case["kind"] == "gesv_batch":
        A = torch.rand(oa[-1], dtype=dt, device=DEV, generator=g).mul_(2).sub_(1)
    else:
        A = torch.empty(oa[-1], dtype=dt, device=DEV)
        F = _normal((oa[-1],), g, dt)
        for i, n in enumerate(ns):
            f = F[oa[i]:oa[i + 1]].view(n, n)
            a = A[oa[i]:oa[i + 1]].view(n, n)
            torch.mm(f, f.T, out=a)
            a.div_(n).diagonal().add_(0.1)
    return ns, rs, oa, ob, A, B


def _pointers(t, off):
    base, size = t.data_ptr(), t.element_size()
    return (C.c_void_p * (len(off) - 1))(*[base + size * o for o in off[:-1]])


def _ints(v):
    return (C.c_int * len(v))(*v)


def _values(case, seed):
    """The inputs of a single-matrix case as tensors in the layout above."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "chol":
        return {"A": _tri(_spd(case["n"], g), case["uplo"])}
    if kind == "spd_solve":
        return {"A": _tri(_spd(case["n"], g), case["uplo"]),
                "B": _normal((case["nrhs"], case["n"]), g)}
    if kind == "lu":
        return {"A": _general(case["m"], case["n"], g)}
    if kind == "lu_solve":
        return {"A": _general(case["n"], case["n"], g),
                "B": _normal((case["nrhs"], case["n"]), g)}
    if kind == "mixed":
        return {"A": _spd_kappa(case["n"], case["kappa"], g),
                "B": _normal((case["nrhs"], case["n"]), g)}
    # chol_solve, adjoint: a lower factor with the entries' sizes of that of B B'/n + I
    n = case["n"]
    L = torch.tril(_normal((n, n), g).div_(math.sqrt(n)))
    L.diagonal().copy_(torch.linspace(2.0, 1.0, n, dtype=torch.float64, device=DEV).sqrt())
    if kind == "chol_solve":
        L = L.T.contiguous() if case["uplo"] == "lower" else L
        return {"L": L, "B": _normal((case["nrhs"], n), g)}
    return {"L": L.T.contiguous(), "Lbar": torch.triu(_normal((n, n), g))}


# ---- the passes --------------------------------------------------------------

def prepare(case, seed):
    fla.FLA_Init()
    s = {"case": case}
    kind = case["kind"]
    if kind in ("posv_batch", "gesv_batch"):
        ns, rs, oa, ob, A, B = _batch_values(case, seed)
        s["A0"], s["B0"], s["A"], s["B"] = A, B, torch.empty_like(A), torch.empty_like(B)
        s["info"] = torch.zeros(len(ns), dtype=torch.int32, device=DEV)
        s["n"], s["nrhs"] = _ints(ns), _ints(rs)
        s["pA"], s["pB"] = _pointers(s["A"], oa), _pointers(s["B"], ob)
        if kind == "gesv_batch":
            op = _offsets(ns)
            s["piv"] = torch.zeros(op[-1], dtype=torch.int32, device=DEV)
            s["pP"] = _pointers(s["piv"], op)
        return s
    v = _values(case, seed)
    s.update({k: Matrix(t) for k, t in v.items()})
    if kind in ("chol", "spd_solve", "lu", "lu_solve"):
        s["F"] = Matrix(torch.zeros_like(v["A"]))
        s["Fo"] = s["F"].obj()
    if kind in ("lu", "lu_solve"):
        p = torch.zeros(1, min(s["A"].m, s["A"].n), dtype=torch.int32, device=DEV)
        s["p"] = Matrix(p)
        s["po"] = s["p"].obj()
    if kind in ("chol_solve", "adjoint"):
        s["Lo"] = s["L"].obj()
    if "B" in s:
        s["X"] = Matrix(torch.zeros_like(v["B"]))
        s["Bo"], s["Xo"] = s["B"].obj(), s["X"].obj()
    if kind == "adjoint":
        s["Lbo"] = s["Lbar"].obj()
        s["Abar"] = Matrix(torch.zeros_like(v["L"]))
        s["Abo"] = s["Abar"].obj()
    return s


def _copy(dst, src, uplo):
    fla.check(fla.lib().fla_hip_dlacpy(uplo, src.m, src.n, src.ptr, src.ld, dst.ptr, dst.ld))


def _copy_flat(dst, src):
    fla.check(fla.lib().fla_hip_memcpy_d2d(dst.data_ptr(), src.data_ptr(),
                                           src.numel() * src.element_size()))


def run(state):
    s = state
    case = s["case"]
    kind = case["kind"]
    if kind in ("chol", "spd_solve"):
        uplo = UPLO[case["uplo"]]
        _copy(s["F"], s["A"], uplo)
        info = fla.FLA_Chol(uplo, s["Fo"])
        if kind == "chol":
            return {"L": s["F"].t, "info": info}
        fla.FLA_Chol_solve(uplo, s["Fo"], s["Bo"], s["Xo"])
        return {"L": s["F"].t, "X": s["X"].t, "info": info}
    if kind in ("lu", "lu_solve"):
        _copy(s["F"], s["A"], fla.FLA_FULL_MATRIX)
        info = fla.FLA_LU_piv(s["Fo"], s["po"])
        if kind == "lu":
            return {"LU": s["F"].t, "p": s["p"].t, "info": info}
        fla.FLA_LU_piv_solve(s["Fo"], s["po"], s["Bo"], s["Xo"])
        return {"LU": s["F"].t, "p": s["p"].t, "X": s["X"].t, "info": info}
    if kind == "chol_solve":
        fla.FLA_Chol_solve(UPLO[case["uplo"]], s["Lo"], s["Bo"], s["Xo"])
        return {"X": s["X"].t}
    if kind == "adjoint":
        fla.FLA_Chol_adjoint(LOWER, s["Lo"], s["Lbo"], s["Abo"])
        return {"Abar": s["Abar"].t}
    if kind == "mixed":
        _, info, _ = fla.dsposv(LOWER, s["A"], s["B"], s["X"])
        return {"X": s["X"].t, "info": info}
    L = fla.lib()
    _copy_flat(s["A"], s["A0"])
    _copy_flat(s["B"], s["B0"])
    info = C.c_void_p(s["info"].data_ptr())
    count = C.c_int(len(s["n"]))
    if kind == "gesv_batch":
        fla.check(L.fla_hip_dgesv_batched(count, s["n"], s["pA"], s["n"], s["pP"], s["pB"], s["n"],
                                          s["nrhs"], info), "dgesv_batched")
        return {"A": s["A"], "X": s["B"], "piv": s["piv"], "info": s["info"]}
    f = L.fla_hip_sposv_batched if case["dtype"] == "f32" else L.fla_hip_dposv_batched
    fla.check(f(count, s["n"], s["pA"], s["n"], s["pB"], s["n"], s["nrhs"], info), "posv_batched")
    return {"A": s["A"], "X": s["B"], "info": s["info"]}


# ---- what the passes have to move and compute, and their results in FP64 -------

def work(case):
    kind = case["kind"]
    if kind in ("posv_batch", "gesv_batch"):
        ns, rs = _batch_shape(case)
        size = 4 if case.get("dtype") == "f32" else 8
        lu = kind == "gesv_batch"
        flops = sum((2 if lu else 1) * n ** 3 / 3 + 2 * n * n * r for n, r in zip(ns, rs))
        move = sum((2 * n * n if lu else n * (n + 1)) + 2 * n * r for n, r in zip(ns, rs))
        return {"bytes": size * move, "flops": flops}
    n = case["n"]
    r = case.get("nrhs", 0)
    if kind == "chol":
        return {"bytes": 8 * n * (n + 1), "flops": n ** 3 / 3}
    if kind == "spd_solve":
        return {"bytes": 8 * n * (n + 1) + 16 * n * r, "flops": n ** 3 / 3 + 2 * n * n * r}
    if kind in ("lu", "lu_solve"):
        m = case.get("m", n)
        k = min(m, n)
        f = 2 * (m * n * k - (m + n) * k * k / 2 + k ** 3 / 3) + 2 * n * n * r
        return {"bytes": 16 * m * n + 16 * n * r, "flops": f}
    if kind == "chol_solve":
        return {"bytes": 4 * n * (n + 1) + 16 * n * r, "flops": 2 * n * n * r}
    if kind == "mixed":
        return {"bytes": 4 * n * (n + 1) + 16 * n * r, "flops": n ** 3 / 3 + 4 * n * n * r}
    # adjoint: L' Lbar (n^3/3) and two triangular solves (n^3 each); two
    # triangles read, the full matrix written
    return {"bytes": 8 * n * (n + 1) + 8 * n * n, "flops": 7 * n ** 3 / 3}


def _exact_batch(case, seed):
    ns, rs, oa, ob, A, B = _batch_values(case, seed)
    A, B = A.double().cpu(), B.double().cpu()
    lu = case["kind"] == "gesv_batch"
    for i, (n, r) in enumerate(zip(ns, rs)):
        a = A[oa[i]:oa[i + 1]].view(n, n)      # a.T is the matrix
        b = B[ob[i]:ob[i + 1]].view(r, n)
        if lu:
            f, p = torch.linalg.lu_factor(a.T)
            b.copy_(torch.linalg.lu_solve(f, p, b.T).T)
            a.copy_(f.T)
        else:
            f = torch.linalg.cholesky(a.T)
            b.copy_(torch.cholesky_solve(b.T, f).T)
            a.copy_(torch.triu(f.T) + torch.tril(a, -1))  # the other triangle is not touched
    return {"A": A, "X": B, "info": None, **({"piv": None} if lu else {})}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("posv_batch", "gesv_batch"):
        return _exact_batch(case, seed)
    v = _values(case, seed)
    if case["n"] <= 16384:                        # beyond, the host would take too long
        v = {k: t.cpu() for k, t in v.items()}
    if kind in ("chol", "spd_solve"):
        # cholesky reads the lower triangle: t for "upper" storage, t.T for "lower"
        low = case["uplo"] == "lower"
        F = torch.linalg.cholesky(v["A"].T if low else v["A"])
        out = {"L": F.T.contiguous() if low else F, "info": None}
        if kind == "spd_solve":
            out["X"] = torch.cholesky_solve(v["B"].T, F).T.contiguous()
        return out
    if kind in ("lu", "lu_solve"):
        F, p = torch.linalg.lu_factor(v["A"].T)
        out = {"LU": F.T.contiguous(), "p": None, "info": None}
        if kind == "lu_solve":
            out["X"] = torch.linalg.lu_solve(F, p, v["B"].T).T.contiguous()
        return out
    if kind == "mixed":
        F = torch.linalg.cholesky(v["A"])
        return {"X": torch.cholesky_solve(v["B"].T, F).T.contiguous(), "info": None}
    if kind == "chol_solve":
        F = v["L"].T if case["uplo"] == "lower" else v["L"]
        return {"X": torch.cholesky_solve(v["B"].T, F).T.contiguous()}
    L = v["L"].T                                  # lower
    P = torch.tril(L.T @ v["Lbar"].T)
    P.diagonal().mul_(0.5)
    Y = torch.linalg.solve_triangular(L.T, P, upper=True)
    G = torch.linalg.solve_triangular(L, Y, upper=False, left=False)
    return {"Abar": (G + G.T) / 2}
