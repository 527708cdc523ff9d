"""GPU tests of how often the factorizations round, against long double: the
factor of one tile, where little is subtracted from the matrix (G G^H / n + I).
A FP64 reference is no better than the library's own results there.

Bounds.  Tile of order 128: an entry is rounded at its own size once for each of
up to 7 block columns of 16 before its own, and inside that one once per column
(real, 7.5 on average) or once (complex): with 0.4 u a rounding 0.4 sqrt(11) =
1.3 u and 0.4 sqrt(4.5) = 0.85 u.  Means over a few matrices each.
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
