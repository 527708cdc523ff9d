"""GPU tests of the complex diagonal-tile kernel for tiles of order <= 128
(one tile factored and inverted in LDS): edge orders of its 16-column panels,
both storages and precisions, and the pivot at which a non positive definite
tile fails.

Bounds: the factor of a well-conditioned matrix of order n has a relative
error of a small multiple of sqrt(n) u; 4 sqrt(n) u is used (u = 2^-53,
2^-24).
The inverse is checked through the solve, whose scaled residual
||b - A x|| / (n ||A|| ||x||) stays below 10 u.
"""
import numpy as np
import pytest

import plasma_amd as pa
from tests import _util as U

pytestmark = pytest.mark.gpu

L, Up = pa.PlasmaLower, pa.PlasmaUpper
DT = {"z": np.complex128, "c": np.complex64}
EPS = {"z": U.EPS64, "c": U.EPS32}


def _hpd(n, seed):
    rng = np.random.default_rng(seed)
    G = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    return G @ G.conj().T / n + 2 * np.eye(n)


def _tile(nb=128):
    pa.set_param(pa.PlasmaTuning, pa.PlasmaDisabled)
    pa.set_param(pa.PlasmaNb, nb)


@pytest.mark.parametrize("prec", ["z", "c"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,nb", [(1, 128), (15, 128), (16, 128), (17, 128),
                                  (33, 128), (100, 128), (127, 128),
                                  (128, 128), (129, 128), (250, 100),
                                  (75, 40)])
def test_factor_and_inverse(plasma, nb_guard, prec, uplo, n, nb):
    _tile(nb)
    A = _hpd(n, n).astype(DT[prec])
    rng = np.random.default_rng(2)
    B = (rng.standard_normal((n, 3)) +
         1j * rng.standard_normal((n, 3))).astype(DT[prec])
    # the imaginary part of the diagonal and the other triangle are not read
    a = A + 1j * np.diag(np.arange(1, n + 1)).astype(DT[prec])
    a = (np.tril(a) if uplo == L else np.triu(a)).astype(DT[prec], order="F")
    b = B.copy(order="F")
    assert pa.posv(uplo, n, 3, a, n, b, n, prec=prec) == 0
    A = A.astype(np.complex128)
    ref = np.linalg.cholesky(A)
    got = np.tril(a) if uplo == L else np.triu(a).conj().T
    assert np.all(np.diag(got).imag == 0)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= 4 * np.sqrt(n) * EPS[prec], err
    assert not np.any(np.triu(a, 1) if uplo == L else np.tril(a, -1))
    r = np.abs(B - A @ b).sum(1).max()
    res = r / (n * np.abs(A).sum(1).max() * np.abs(b).sum(1).max())
    assert res <= 10 * EPS[prec], res


@pytest.mark.parametrize("prec", ["z", "c"])
@pytest.mark.parametrize("col", [0, 15, 16, 77, 127])
@pytest.mark.parametrize("value", [0.0, -1.0, np.nan])
def test_failed_pivot(plasma, nb_guard, prec, col, value):
    _tile()
    A = np.asfortranarray(np.eye(128, dtype=DT[prec]) * 4)
    A[col, col] = value
    a = A.copy(order="F")
    assert pa.potrf(L, 128, a, 128, prec=prec) == col + 1
    assert np.array_equal(a, A, equal_nan=True)
