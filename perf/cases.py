"""Workloads of the Cholesky solve path, as a user's program calls it, for
timing and for comparing results: single solves in every precision, the
mixed-precision solver, batches of small systems, the inverse, and the
Gaussian-process log-likelihood with its gradient.

All arrays live in device memory.  The library runs on its own streams, so
a program that prepares arrays with torch waits for torch's stream before it
calls in; the library's calls return when their results are in place.  A
matrix that a routine overwrites is a copy of the caller's, as a program
makes that still needs its matrix afterwards (the next right-hand side, the
residual, the next step of an optimizer).

Column-major arrays are torch tensors of the transposed shape: element
(i, j) of a matrix is T[j, i].
"""
import ctypes
import math

import numpy as np
import torch

import plasma_amd as pa

REAL = {"d": torch.float64, "s": torch.float32,
        "z": torch.float64, "c": torch.float32}
DTYPE = {"d": torch.float64, "s": torch.float32,
         "z": torch.complex128, "c": torch.complex64}
ELEM = {"d": 8, "s": 4, "z": 16, "c": 8}


def listed():
    return [
        # one small system with one right-hand side, e.g. a Newton step or
        # a small least-squares problem: latency and launches
        {"name": "dposv_n500", "kind": "posv", "prec": "d", "n": 500,
         "nrhs": 1, "uplo": "L", "graph": False},
        # a moderate system of odd order with a partial last tile, upper
        # storage, a few right-hand sides
        {"name": "dposv_n2049", "kind": "posv", "prec": "d", "n": 2049,
         "nrhs": 10, "uplo": "U", "graph": False},
        # the ordinary dense solve, the same order again and again, so with
        # captured launches
        {"name": "dposv_n8192", "kind": "posv", "prec": "d", "n": 8192,
         "nrhs": 64, "uplo": "L", "graph": True},
        # a large double precision solve
        {"name": "dposv_n16384", "kind": "posv", "prec": "d", "n": 16384,
         "nrhs": 64, "uplo": "L", "graph": False},
        # single precision, upper storage, order no multiple of the tile
        {"name": "sposv_n6000", "kind": "posv", "prec": "s", "n": 6000,
         "nrhs": 16, "uplo": "U", "graph": False},
        # mixed precision at a moderate order, few right-hand sides
        {"name": "dsposv_n4000", "kind": "dsposv", "n": 4000, "nrhs": 8,
         "uplo": "L", "kappa": 1e4, "graph": False},
        # the headline: mixed precision at n = 32768, condition 1e6
        {"name": "dsposv_n32768", "kind": "dsposv", "n": 32768, "nrhs": 64,
         "uplo": "L", "kappa": 1e6, "graph": True},
        # complex Hermitian solve (frequency-domain problems), ragged
        {"name": "zposv_n5001", "kind": "posv", "prec": "z", "n": 5001,
         "nrhs": 32, "uplo": "L", "graph": False},
        # many independent systems of uneven order, one right-hand side
        # (local Gaussian processes)
        {"name": "batched_d", "kind": "batched", "prec": "d", "count": 1024,
         "nmin": 32, "nmax": 512, "nrhs": 1, "uplo": "L", "noise": 1e-3},
        # very many small systems in single precision
        {"name": "batched_s_small", "kind": "batched", "prec": "s",
         "count": 4096, "nmin": 8, "nmax": 128, "nrhs": 1, "uplo": "L",
         "noise": 1e-2},
        # one step of a Gaussian process's hyperparameter fit: factor,
        # solve, log-likelihood and its gradient with respect to the kernel
        # matrix (forward and backward)
        {"name": "gp_d_n4096", "kind": "gp", "prec": "d", "n": 4096},
        # the inverse of a covariance matrix
        {"name": "dpoinv_n3000", "kind": "poinv", "prec": "d", "n": 3000,
         "uplo": "L"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["posv"] * 5 + ["dsposv"] * 3 + ["batched"] * 2 +
                      ["gp", "poinv"])
    uplo = rng.choice("LU")
    if kind == "posv":
        prec = rng.choice("dddssz")
        return {"kind": kind, "prec": prec,
                "n": _log_int(rng, 100, 6000 if prec == "z" else 16384),
                "nrhs": _log_int(rng, 1, 100), "uplo": uplo,
                "graph": rng.random() < 0.3}
    if kind == "dsposv":
        return {"kind": kind, "n": _log_int(rng, 500, 32768),
                "nrhs": _log_int(rng, 1, 64), "uplo": uplo,
                "kappa": rng.choice([1e2, 1e4, 1e6]),
                "graph": rng.random() < 0.5}
    if kind == "batched":
        prec = rng.choice("ds")
        nmax = _log_int(rng, 48, 512)
        return {"kind": kind, "prec": prec,
                "count": _log_int(rng, 64, min(4096, 1024 * 512 // nmax)),
                "nmin": rng.randint(1, nmax // 2), "nmax": nmax,
                "nrhs": rng.choice([1, 1, 2, 5]), "uplo": uplo,
                "noise": 1e-3 if prec == "d" else 1e-2}
    if kind == "gp":
        return {"kind": kind, "prec": rng.choice("ds"),
                "n": _log_int(rng, 300, 8192)}
    return {"kind": kind, "prec": rng.choice("ds"),
            "n": _log_int(rng, 200, 6000), "uplo": uplo}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 11)


def _randn(shape, dtype, g):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=g)


def _ggt(n, prec, g):
    """G G^H / n + I, G iid N(0, 1) entries (E|g|^2 = 1 if complex)."""
    if prec in "ds":
        G = _randn((n, n), torch.float64, g)
        A = (G @ G.T).div_(n)
    else:
        G = torch.complex(_randn((n, n), torch.float64, g),
                          _randn((n, n), torch.float64, g))
        A = (G @ G.mH).div_(2 * n)
        A = (A + A.mH) * 0.5
    A.diagonal().add_(1.0)
    return A.to(DTYPE[prec])


def _householder(n, kappa, g, nrefl=64):
    """(V, tau, s): Q = H_1 ... H_k with H_i = I - tau_i v_i v_i^T from
    N(0, 1) vectors, and eigenvalues log-spaced on [1 / kappa, 1]."""
    nrefl = min(nrefl, n)
    V = _randn((nrefl, n), torch.float64, g)
    tau = 2.0 / (V * V).sum(1)
    i = torch.arange(n, dtype=torch.float64, device="cuda")
    s = torch.exp(-math.log(kappa) * i / max(n - 1, 1))
    return V, tau, s


def _householder_matrix(V, tau, s):
    """Q diag(s) Q^T through the compact form Q = I - V^T T V."""
    k, n = V.shape
    gram, tau = (V @ V.T).cpu(), tau.cpu()
    T = torch.zeros(k, k, dtype=torch.float64)
    for j in range(k):
        T[j, j] = tau[j]
        if j:
            T[:j, j] = -tau[j] * (T[:j, :j] @ gram[:j, j])
    U = V * s
    C = T @ (V @ U.T).cpu() @ T.T
    M = torch.zeros(2 * k, 2 * k, dtype=torch.float64)
    M[:k, :k], M[:k, k:], M[k:, :k] = C, -T, -T.T
    W = torch.cat([V, U])
    A = W.T @ (M.cuda() @ W)
    A.diagonal().add_(s)
    return (A + A.T).mul_(0.5)


def _gp_matrix(n, prec, g):
    """RBF kernel of lengthscale 1 on n points ~ N(0, 1)^8, plus 0.1 I."""
    X = _randn((n, 8), torch.float64, g)
    sq = (X * X).sum(1)
    D2 = (sq[:, None] + sq[None, :] - 2.0 * (X @ X.T)).clamp_min_(0.0)
    K = torch.exp(-0.5 * D2)
    K = (K + K.T) * 0.5
    K.diagonal().fill_(1.1)
    return K.to(DTYPE[prec])


def _batch_sizes(case):
    """The orders of a batch's systems: the case's, for every seed."""
    return np.random.default_rng(case["count"]).integers(
        case["nmin"], case["nmax"] + 1, case["count"]).astype(np.int32)


def _batch_mask(n, nmax):
    k = torch.from_numpy(n).cuda()[:, None]
    return torch.arange(nmax, device="cuda")[None, :] < k


def _batch_padded(case, seed):
    """The systems padded to the largest order with the identity: kernel
    matrices exp(-|x - y|^2 / (2 0.2^2)) of points ~ U[0, 1]^3 + noise I,
    with right-hand sides ~ N(0, 1); and the mask of valid rows."""
    g = _gen(seed)
    n = _batch_sizes(case)
    nmax = int(n.max())
    ok = _batch_mask(n, nmax)
    x = torch.rand((case["count"], nmax, 3), dtype=torch.float64,
                   device="cuda", generator=g)
    K = torch.zeros((case["count"], nmax, nmax), dtype=torch.float64,
                    device="cuda")
    for d in range(3):
        K -= (x[:, :, None, d] - x[:, None, :, d]).square_()
    K.div_(2 * 0.2 ** 2).exp_()
    K.diagonal(dim1=1, dim2=2).add_(case["noise"])
    K = K.to(DTYPE[case["prec"]])
    B = _randn((case["count"], case["nrhs"], nmax), DTYPE[case["prec"]], g)
    return n, ok, K, B


def prepare(case, seed):
    pa.load().plasma_init()      # says so when it is initialised already
    pa.set_param(pa.PlasmaGraphCapture,
                 pa.PlasmaEnabled if case.get("graph")
                 else pa.PlasmaDisabled)
    g = _gen(seed)
    kind = case["kind"]
    st = {"case": case, "uplo": pa.PlasmaUpper if case.get("uplo") == "U"
          else pa.PlasmaLower}
    if kind == "posv":
        st["A"] = _ggt(case["n"], case["prec"], g)
        st["B"] = _randn((case["nrhs"], case["n"]), DTYPE[case["prec"]], g)
        st["F"], st["X"] = torch.empty_like(st["A"]), torch.empty_like(st["B"])
    elif kind == "dsposv":
        st["A"] = _householder_matrix(*_householder(case["n"], case["kappa"],
                                                    g))
        st["B"] = _randn((case["nrhs"], case["n"]), torch.float64, g)
        st["X"] = torch.empty_like(st["B"])
    elif kind == "batched":
        n, ok, K, B = _batch_padded(case, seed)
        st["A"] = torch.masked_select(K, ok[:, :, None] & ok[:, None, :])
        st["B"] = torch.masked_select(B, ok[:, None, :])
        st["n"] = n
        n64 = n.astype(np.uint64)
        st["aoff"] = np.concatenate([[0], np.cumsum(n64 * n64)[:-1]]).astype(
            np.uint64)
        st["boff"] = np.concatenate(
            [[0], np.cumsum(n64 * np.uint64(case["nrhs"]))[:-1]]).astype(
                np.uint64)
        st["F"], st["X"] = torch.empty_like(st["A"]), torch.empty_like(st["B"])
        st["info"] = np.zeros(case["count"], dtype=np.int32)
    elif kind == "gp":
        st["A"] = _gp_matrix(case["n"], case["prec"], g)
        st["B"] = _randn((1, case["n"]), DTYPE[case["prec"]], g)
        st["F"], st["G"] = torch.empty_like(st["A"]), torch.empty_like(st["A"])
        st["X"], st["Y"] = torch.empty_like(st["B"]), torch.empty_like(st["B"])
    else:
        st["A"] = _ggt(case["n"], case["prec"], g)
        st["F"] = torch.empty_like(st["A"])
    torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _check(rc):
    if rc != 0:
        raise RuntimeError("the library returned %d" % rc)


def run(st):
    case = st["case"]
    kind, prec, uplo = case["kind"], case.get("prec"), st["uplo"]
    wait = torch.cuda.current_stream().synchronize
    if kind == "posv":
        n, nrhs = case["n"], case["nrhs"]
        st["F"].copy_(st["A"])
        st["X"].copy_(st["B"])
        wait()
        _check(pa.posv(uplo, n, nrhs, st["F"], n, st["X"], n, prec=prec))
        return {"factor": st["F"], "x": st["X"]}
    if kind == "dsposv":
        n, nrhs = case["n"], case["nrhs"]
        rc, _ = pa.dsposv(uplo, n, nrhs, st["A"], n, st["B"], n, st["X"], n)
        _check(rc)
        return {"x": st["X"]}
    if kind == "batched":
        st["F"].copy_(st["A"])
        st["X"].copy_(st["B"])
        wait()
        fn = getattr(pa.load(), "plasma_%sposv_vbatched" % prec)
        _check(fn(uplo, case["count"], st["n"].ctypes.data,
                  st["F"].data_ptr(), st["aoff"].ctypes.data, case["nrhs"],
                  st["X"].data_ptr(), st["boff"].ctypes.data,
                  st["info"].ctypes.data))
        return {"factor": st["F"], "x": st["X"], "info": st["info"]}
    if kind == "gp":
        n, F, G, X, Y = case["n"], st["F"], st["G"], st["X"], st["Y"]
        F.copy_(st["A"])
        X.copy_(st["B"])
        wait()
        _check(pa.potrf(uplo, n, F, n, prec=prec))
        _check(pa.potrs(uplo, n, 1, F, n, X, n, prec=prec))
        d = F.diagonal()
        loglik = -0.5 * (st["B"] * X).sum() - d.log().sum()
        # the adjoints of the factor (from log det) and of the solution
        G.zero_()
        G.diagonal().copy_(-1.0 / d)
        torch.mul(st["B"], -0.5, out=Y)
        wait()
        _check(pa.potrf_adjoint(uplo, n, F, n, G, n, prec=prec))
        _check(pa.potrs_adjoint(uplo, n, 1, F, n, X, n, Y, n, G, n,
                                prec=prec))
        return {"alpha": X, "loglik": loglik, "grad": G}
    n = case["n"]
    st["F"].copy_(st["A"])
    wait()
    fn = getattr(pa.load(), "plasma_%spoinv" % prec)
    _check(fn(uplo, n, st["F"].data_ptr(), n))
    return {"inverse": st["F"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and what its results are
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "batched":
        n = _batch_sizes(case).astype(np.float64)
        nrhs, es = case["nrhs"], ELEM[case["prec"]]
        return {"bytes": float((2 * n * n + 2 * n * nrhs).sum()) * es,
                "flops": float((n ** 3 / 3 + 2 * n * n * nrhs).sum())}
    n = float(case["n"])
    if kind == "dsposv":
        return {"bytes": (n * n + 2 * n * case["nrhs"]) * 8,
                "flops": n ** 3 / 3 + 2 * n * n * case["nrhs"]}
    es = ELEM[case["prec"]]
    if kind == "posv":
        f = n ** 3 / 3 + 2 * n * n * case["nrhs"]
        return {"bytes": (2 * n * n + 2 * n * case["nrhs"]) * es,
                "flops": f * (4 if case["prec"] in "zc" else 1)}
    if kind == "gp":
        # factor n^3/3, adjoint of the factor 2 n^3/3, two solves
        return {"bytes": (2 * n * n + 2 * n) * es, "flops": n ** 3 + 6 * n * n}
    return {"bytes": 2 * n * n * es, "flops": n ** 3}


def tolerance(case):
    """About four times the largest error against 64-bit results that was
    measured over the declared ranges; for the mixed solver the forward
    error that its stopping test admits (a backward error of eps sqrt(n),
    2e-14 at n = 32768, times the condition number, twice)."""
    if case["kind"] == "dsposv":
        return {"rel": 4e-14 * case["kappa"]}
    single = case["prec"] in "sc"
    if case["kind"] == "batched":
        return {"rel": 1e-4 if single else 1e-11}
    if case["kind"] == "gp":
        return {"rel": 4e-5 if single else 1e-13}
    return {"rel": 1e-5 if single else 2e-14}


def _merge(T, tri, upper):
    """T with the stored triangle of its matrix replaced.  `tri` is the
    lower triangular matrix L of the matrix A = L L^H that T holds."""
    if upper:       # U = L^H at T[j, i], i <= j: the lower triangle of T
        return torch.tril(tri.conj()) + torch.triu(T, 1)
    return torch.triu(tri.mT) + torch.tril(T, -1)


def exact(case, seed):
    kind, upper = case["kind"], case.get("uplo") == "U"
    g = _gen(seed)
    if kind == "posv":
        T = _ggt(case["n"], case["prec"], g)
        B = _randn((case["nrhs"], case["n"]), DTYPE[case["prec"]], g)
        wide = torch.complex128 if T.is_complex() else torch.float64
        T, B = T.to(wide), B.to(wide)
        L = torch.linalg.cholesky(T.mT.contiguous())
        X = torch.cholesky_solve(B.mT.contiguous(), L)
        return {"factor": _merge(T, L, upper), "x": X.mT}
    if kind == "dsposv":
        V, tau, s = _householder(case["n"], case["kappa"], g)
        if case["n"] <= 8192:
            L = torch.linalg.cholesky(_householder_matrix(V, tau, s))
            B = _randn((case["nrhs"], case["n"]), torch.float64, g)
            return {"x": torch.cholesky_solve(B.mT.contiguous(), L).mT}
        # A^-1 = Q diag(1 / s) Q^T, the reflectors one by one
        X = _randn((case["nrhs"], case["n"]), torch.float64, g)
        for v, t in zip(V, tau):
            X -= t * torch.outer(X @ v, v)
        X /= s
        for v, t in zip(V.flip(0), tau.flip(0)):
            X -= t * torch.outer(X @ v, v)
        return {"x": X}
    if kind == "batched":
        n, ok, K, B = _batch_padded(case, seed)
        m = ok[:, :, None] & ok[:, None, :]
        T = torch.where(m, K.double(), torch.eye(
            K.shape[1], dtype=torch.float64, device="cuda"))
        L = torch.linalg.cholesky(T)
        X = torch.cholesky_solve(
            torch.where(ok[:, None, :], B.double(), 0.0).mT.contiguous(), L)
        return {"factor": torch.masked_select(_merge(T, L, upper), m),
                "x": torch.masked_select(X.mT, ok[:, None, :]),
                "info": None}
    if kind == "gp":
        K = _gp_matrix(case["n"], case["prec"], g).double()
        y = _randn((1, case["n"]), DTYPE[case["prec"]], g).double()
        L = torch.linalg.cholesky(K)
        a = torch.cholesky_solve(y.mT.contiguous(), L).mT
        loglik = -0.5 * (y * a).sum() - L.diagonal().log().sum()
        grad = 0.5 * (a.mT @ a - torch.cholesky_inverse(L))
        return {"alpha": a, "loglik": loglik, "grad": grad}
    T = _ggt(case["n"], case["prec"], g).double()
    inv = torch.cholesky_inverse(torch.linalg.cholesky(T))
    inv = (inv + inv.mT) * 0.5
    return {"inverse": _merge(T, inv, upper)}
