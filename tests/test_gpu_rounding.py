"""GPU tests of how often the factorizations round, against long double: the
factor of one tile, where little is subtracted from the matrix (G G^H / n + I),
and factors of kernel (RBF) matrices, whose trailing blocks nearly cancel.  A
FP64 reference is no better than the library's own results there.

Bounds.  Tile of order 128: an entry is rounded at its own size once for each of
up to 7 block columns of 16 before its own, and inside that one once per column
(real, 7.5 on average) or once (complex): with 0.4 u a rounding 0.4 sqrt(11) =
1.3 u and 0.4 sqrt(4.5) = 0.85 u.  Kernel matrices: 1.5 times the error of a
factorization by block columns of 32 in NumPy, which subtracts the product of 32
columns as a whole.  Means over a few matrices each.
"""
import numpy as np
import pytest

import plasma_amd as pa

pytestmark = pytest.mark.gpu

L, Up = pa.PlasmaLower, pa.PlasmaUpper
DT = {"d": np.float64, "s": np.float32, "z": np.complex128,
      "c": np.complex64}


def _exact(A):
    F = A.astype(np.clongdouble if np.iscomplexobj(A) else np.longdouble)
    for j in range(len(F)):
        F[j, j] = np.sqrt(F[j, j].real)
        F[j + 1:, j] /= F[j, j]
        F[j + 1:, j + 1:] -= np.outer(F[j + 1:, j], F[j + 1:, j].conj())
    return np.tril(F)


def _error(F, ref):
    """||F - ref|| / ||ref|| in units of F's u"""
    norm = lambda x: np.sqrt(float((np.abs(x) ** 2).sum()))
    return norm(F - ref) / norm(ref) / (np.finfo(F.dtype).eps / 2)


def _lower(a, uplo):
    return np.tril(a) if uplo == L else np.triu(a).conj().T


@pytest.mark.parametrize("prec,limit", [("d", 1.3), ("s", 1.3), ("z", 0.85),
                                        ("c", 0.85)])
@pytest.mark.parametrize("uplo", [L, Up])
def test_tile(plasma, nb_guard, prec, limit, uplo):
    n = 128
    pa.set_param(pa.PlasmaNb, n)
    err = []
    for seed in range(4):
        rng = np.random.default_rng(seed)
        G = rng.standard_normal((n, n))
        if prec in "zc":
            G = G + 1j * rng.standard_normal((n, n))
        A = (G @ G.conj().T / n / (2 if prec in "zc" else 1) +
             np.eye(n)).astype(DT[prec])
        A = np.tril(A, -1)
        A = A + A.conj().T + 2 * np.eye(n, dtype=DT[prec])
        a = np.asfortranarray(A)
        assert pa.potrf(uplo, n, a, n, prec=prec) == 0
        err.append(_error(_lower(a, uplo), _exact(A)))
    assert np.mean(err) <= limit, err


def _rbf(n, seed, noise=1e-3):
    X = np.random.default_rng(seed).standard_normal((n, 8))
    D2 = sum((X[:, i, None] - X[None, :, i]) ** 2 for i in range(8))
    return np.exp(-D2 / 8) + noise * np.eye(n)


def _by_32_columns(A):
    F = A.copy()
    for j in range(0, len(F), 32):
        k = j + 32
        F[j:k, j:k] = np.linalg.cholesky(F[j:k, j:k])
        F[k:, j:k] = np.linalg.solve(F[j:k, j:k], F[k:, j:k].T).T
        F[k:, k:] -= F[k:, j:k] @ F[k:, j:k].T
    return np.tril(F)


@pytest.mark.parametrize("uplo", [L, Up])
def test_posv_kernel_matrix(plasma, nb_guard, uplo):
    n = 512
    pa.set_param(pa.PlasmaNb, 128)
    err, lim = [], []
    for seed in range(3):
        A = _rbf(n, seed)
        ref = _exact(A)
        a = np.asfortranarray(A)
        assert pa.potrf(uplo, n, a, n) == 0
        err.append(_error(_lower(a, uplo), ref))
        lim.append(_error(_by_32_columns(A), ref))
    assert np.mean(err) <= 1.5 * np.mean(lim), (err, lim)


@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n", [128, 250, 400])
def test_batched_kernel_matrix(plasma, uplo, n):
    import torch
    mats = [_rbf(n, seed) for seed in range(4)]
    order = np.full(4, n, dtype=np.int32)
    off = (np.arange(4) * n * n).astype(np.uint64)
    info = np.full(4, -7, dtype=np.int32)
    d = torch.from_numpy(np.concatenate([A.ravel() for A in mats])).cuda()
    torch.cuda.synchronize()
    assert pa.load().plasma_dpotrf_vbatched(
        uplo, 4, order.ctypes.data, d.data_ptr(), off.ctypes.data,
        info.ctypes.data) == 0
    assert not info.any()
    err, lim = [], []
    for A, a in zip(mats, d.cpu().numpy().reshape(4, n, n)):
        ref = _exact(A)
        err.append(_error(_lower(a.T, uplo), ref))
        lim.append(_error(_by_32_columns(A), ref))
    assert np.mean(err) <= 1.5 * np.mean(lim), (err, lim)
