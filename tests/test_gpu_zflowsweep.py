"""GPU tests of the one-launch complex triangular sweeps (posv, potrs): last
tiles of every remainder of the K groups of 4 and around the half tile (64),
tiles below one group, right-hand sides around the groups of 8 and around the
largest count that takes them, both storages and precisions.

Bound: the scaled residual ||B - A X|| / (n ||A|| ||X||) stays below 10 u.
"""
import numpy as np
import pytest

import plasma_amd as pa
from tests import _util as U

pytestmark = pytest.mark.gpu

L, Up = pa.PlasmaLower, pa.PlasmaUpper


def _solve(prec, uplo, n, nrhs, nb, split_calls):
    pa.set_param(pa.PlasmaNb, nb)
    dt = np.complex128 if prec == "z" else np.complex64
    rng = np.random.default_rng(n)
    G = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    A = (G @ G.conj().T / n + 2 * np.eye(n)).astype(dt)
    B = (rng.standard_normal((n, nrhs)) +
         1j * rng.standard_normal((n, nrhs))).astype(dt)
    a = A.copy(order="F")
    b = np.zeros((n + 2, nrhs), dtype=dt, order="F")
    b[:n] = B
    if split_calls:
        assert pa.potrf(uplo, n, a, n, prec=prec) == 0
        assert pa.potrs(uplo, n, nrhs, a, n, b, n + 2, prec=prec) == 0
    else:
        assert pa.posv(uplo, n, nrhs, a, n, b, n + 2, prec=prec) == 0
    A, X = A.astype(np.complex128), b[:n].astype(np.complex128)
    res = np.abs(B - A @ X).sum(1).max() / (
        n * np.abs(A).sum(1).max() * np.abs(X).sum(1).max())
    assert res <= 10 * (U.EPS64 if prec == "z" else U.EPS32), res
    assert not b[n:].any()


@pytest.mark.parametrize("prec", ["z", "c"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("last", [1, 3, 4, 5, 17, 63, 64, 65, 102, 127, 128])
def test_last_tile(plasma, nb_guard, prec, uplo, last):
    _solve(prec, uplo, 256 + last, 5, 128, False)


@pytest.mark.parametrize("prec", ["z", "c"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,nb", [(23, 5), (100, 12), (37, 37), (130, 65),
                                  (1, 128), (9, 128), (7, 3)])
def test_small_tiles(plasma, nb_guard, prec, uplo, n, nb):
    _solve(prec, uplo, n, 3, nb, True)


@pytest.mark.parametrize("prec", ["z", "c"])
@pytest.mark.parametrize("nrhs", [1, 7, 8, 9, 33, 128, 129])
def test_right_hand_sides(plasma, nb_guard, prec, nrhs):
    _solve(prec, L, 300, nrhs, 128, True)
    _solve(prec, Up, 300, nrhs, 100, False)


def test_many_tiles(plasma, nb_guard):
    # more block rows than workgroups the chip holds at once
    _solve("z", L, 1300, 2, 2, False)
