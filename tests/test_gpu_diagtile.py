"""GPU tests of the diagonal-tile kernel for tiles of order <= 128 (one tile
factored and inverted in LDS): edge orders of its 16-column panels, both
storages and precisions, the pivot at which a non positive definite tile
fails, and pivots far from 1.

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
DT = {"d": np.float64, "s": np.float32}
EPS = {"d": U.EPS64, "s": U.EPS32}


def _tile(nb=128):
    pa.set_param(pa.PlasmaTuning, pa.PlasmaDisabled)
    pa.set_param(pa.PlasmaNb, nb)


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,nb", [(1, 128), (15, 128), (16, 128), (17, 128),
                                  (100, 128), (127, 128), (128, 128),
                                  (129, 128), (250, 100), (75, 40)])
def test_factor_and_inverse(plasma, nb_guard, prec, uplo, n, nb):
    _tile(nb)
    A = U.ggt_spd(n, seed=n).astype(DT[prec])
    B = U.rhs(n, 3, seed=2).astype(DT[prec])
    a, b = A.copy(order="F"), B.copy(order="F")
    assert pa.posv(uplo, n, 3, a, n, b, n, prec=prec) == 0
    ref = np.linalg.cholesky(A.astype(np.float64))
    got = np.tril(a) if uplo == L else np.triu(a).T
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= 4 * np.sqrt(n) * EPS[prec], err
    other = np.triu(a, 1) if uplo == L else np.tril(a, -1)
    keep = np.triu(A, 1) if uplo == L else np.tril(A, -1)
    assert np.array_equal(other, keep)
    res = U.scaled_residual(A.astype(np.float64), b.astype(np.float64),
                            B.astype(np.float64))
    assert res <= 10 * EPS[prec], res


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("col", [0, 15, 16, 77, 127])
@pytest.mark.parametrize("value", [0.0, -1.0, np.nan])
def test_failed_pivot(plasma, nb_guard, prec, col, value):
    _tile()
    A = np.asfortranarray(np.eye(128, dtype=DT[prec]) * 4)
    A[col, col] = value
    a = A.copy(order="F")
    assert pa.potrf(L, 128, a, 128, prec=prec) == col + 1
    assert np.array_equal(a, A, equal_nan=True)


@pytest.mark.parametrize("prec,shift", [("d", 900), ("d", -900), ("s", 90),
                                        ("s", -90)])
def test_pivots_far_from_one(plasma, nb_guard, prec, shift):
    # scaling A by 2^shift scales the factor by 2^(shift / 2)
    _tile()
    n = 128
    A = U.ggt_spd(n, seed=4).astype(DT[prec])
    a = np.asfortranarray(np.ldexp(A, shift).astype(DT[prec]))
    assert pa.potrf(L, n, a, n, prec=prec) == 0
    ref = np.linalg.cholesky(A.astype(np.float64))
    got = np.ldexp(np.tril(a).astype(np.float64), -shift // 2)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= 4 * np.sqrt(n) * EPS[prec], err


def test_infinite_pivot(plasma, nb_guard):
    # LAPACK accepts an infinite pivot: its column becomes zero
    _tile()
    A = np.asfortranarray(np.eye(40) * 4.0 + 1.0)
    A[20, 20] = np.inf
    a = A.copy(order="F")
    assert pa.potrf(L, 40, a, 40) == 0
    f = np.tril(a)
    assert np.isinf(f[20, 20]) and np.all(f[21:, 20] == 0)
    assert np.all(np.isfinite(f[21:, 21:]))
