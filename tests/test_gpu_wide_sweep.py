"""GPU tests of the sweeps with many right-hand sides (1024 and more: potrs)
and of the sweep of the identity (poinv): tiles and last tiles that are no
multiple of the 32, 64 and 128 wide blocks, odd strides, few and many tile
rows, both storages and precisions.

Bounds: the scaled residual ||B - A X|| / (n ||A|| ||X||) stays below 10 u;
for the inverse the same with B = I.
"""
import numpy as np
import pytest

import plasma_amd as pa
from tests import _util as U

pytestmark = pytest.mark.gpu

L, Up = pa.PlasmaLower, pa.PlasmaUpper
DT = {"d": np.float64, "s": np.float32}
EPS = {"d": U.EPS64, "s": U.EPS32}


def _nb(nb):
    pa.set_param(pa.PlasmaTuning, pa.PlasmaDisabled)
    pa.set_param(pa.PlasmaNb, nb)


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,nrhs,nb", [(37, 1024, 37), (200, 1025, 100),
                                       (129, 1100, 128), (900, 1024, 65),
                                       (1400, 1030, 256)])
def test_potrs(plasma, nb_guard, prec, uplo, n, nrhs, nb):
    _nb(nb)
    A = U.ggt_spd(n, seed=n).astype(DT[prec])
    B = U.rhs(n, nrhs, seed=n + 1).astype(DT[prec])
    a, b = A.copy(order="F"), B.copy(order="F")
    assert pa.potrf(uplo, n, a, n, prec=prec) == 0
    assert pa.potrs(uplo, n, nrhs, a, n, b, n, prec=prec) == 0
    res = U.scaled_residual(A.astype(np.float64), b.astype(np.float64),
                            B.astype(np.float64))
    assert res <= 10 * EPS[prec], res


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,nb", [(1, 128), (129, 128), (300, 37),
                                  (1023, 128), (1281, 128), (1300, 65),
                                  (1500, 200), (2100, 100)])
def test_inverse(plasma, nb_guard, prec, uplo, n, nb):
    _nb(nb)
    A = U.ggt_spd(n, seed=n).astype(DT[prec])
    a = A.copy(order="F")
    poinv = getattr(pa.load(), "plasma_%spoinv" % prec)
    assert poinv(uplo, n, pa._ptr(a), n) == 0
    low = uplo == L
    X = U.sym_full(a.astype(np.float64), low)
    res = U.scaled_residual(A.astype(np.float64), X, np.eye(n))
    assert res <= 10 * EPS[prec], res
    other = np.triu(a, 1) if low else np.tril(a, -1)
    keep = np.triu(A, 1) if low else np.tril(A, -1)
    assert np.array_equal(other, keep)
