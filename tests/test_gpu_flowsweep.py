"""GPU tests of the one-launch triangular sweeps (posv, potrs): last tiles of
every remainder of the K chunk (8 in FP64, 16 in FP32), tiles below one
chunk, right-hand sides around the groups of 16 and around the largest count
that takes them, both storages and precisions.

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
    dt = np.float64 if prec == "d" else np.float32
    A = U.ggt_spd(n, seed=n).astype(dt)
    B = U.rhs(n, nrhs, seed=n + 1).astype(dt)
    a = A.copy(order="F")
    b = np.zeros((n + 2, nrhs), dtype=dt, order="F")
    b[:n] = B
    if split_calls:
        assert pa.potrf(uplo, n, a, n, prec=prec) == 0
        assert pa.potrs(uplo, n, nrhs, a, n, b, n + 2, prec=prec) == 0
    else:
        assert pa.posv(uplo, n, nrhs, a, n, b, n + 2, prec=prec) == 0
    res = U.scaled_residual(A.astype(np.float64), b[:n].astype(np.float64),
                            B.astype(np.float64))
    assert res <= 10 * (U.EPS64 if prec == "d" else U.EPS32), res
    assert not b[n:].any()


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("last", [1, 3, 7, 8, 9, 15, 16, 17, 40, 101, 127,
                                  128])
def test_last_tile(plasma, nb_guard, prec, uplo, last):
    _solve(prec, uplo, 256 + last, 5, 128, False)


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,nb", [(23, 5), (100, 12), (37, 37), (130, 65),
                                  (1, 128), (9, 128)])
def test_small_tiles(plasma, nb_guard, prec, uplo, n, nb):
    _solve(prec, uplo, n, 3, nb, True)


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("nrhs", [1, 15, 16, 17, 33, 128, 129])
def test_right_hand_sides(plasma, nb_guard, prec, nrhs):
    _solve(prec, L, 300, nrhs, 128, True)
    _solve(prec, Up, 300, nrhs, 100, False)


def test_many_tiles(plasma, nb_guard):
    # more block rows than workgroups the chip holds at once
    n, nb = 3100, 4
    _solve("d", L, n, 2, nb, False)
