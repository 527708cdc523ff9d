"""GPU tests of the complex panel solve and trailing updates: tiles that are
no multiple of the 32 and 64 wide blocks, K that is no multiple of 4 or below
4, ragged last tiles, and tile counts on both sides of the line where the
update moves from its own stream (blocks of 64) to the panel's (blocks of 32).

Bound: the relative error of the factor of a well-conditioned matrix is a
small multiple of sqrt(n) u; 4 sqrt(n) u is used.
"""
import numpy as np
import pytest

import plasma_amd as pa
from tests import _util as U

pytestmark = pytest.mark.gpu

L, Up = pa.PlasmaLower, pa.PlasmaUpper


@pytest.mark.parametrize("prec", ["z", "c"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,nb", [(13, 3), (150, 30), (95, 33), (301, 100),
                                  (22 * 32, 32), (23 * 32, 32),
                                  (26 * 32 + 5, 32), (30 * 30 + 1, 30),
                                  (1200, 65), (700, 200)])
def test_factor(plasma, nb_guard, prec, uplo, n, nb):
    pa.set_param(pa.PlasmaTuning, pa.PlasmaDisabled)
    pa.set_param(pa.PlasmaNb, nb)
    dt = np.complex128 if prec == "z" else np.complex64
    rng = np.random.default_rng(n)
    G = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    A = (G @ G.conj().T / n + 2 * np.eye(n)).astype(dt)
    a = (np.tril(A) if uplo == L else np.triu(A)).copy(order="F")
    assert pa.potrf(uplo, n, a, n, prec=prec) == 0
    ref = np.linalg.cholesky(A.astype(np.complex128))
    got = np.tril(a) if uplo == L else np.triu(a).conj().T
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= 4 * np.sqrt(n) * (U.EPS64 if prec == "z"
                                    else U.EPS32), err
    assert not np.any(np.triu(a, 1) if uplo == L else np.tril(a, -1))
