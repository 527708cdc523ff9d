"""GPU tests on ill-conditioned kernel matrices K = RBF(X) + noise I, whose
diagonal tiles are about as ill-conditioned as the matrix (those of rotation
invariant matrices, as in test_gpu_dsposv.py, are not): the FP32 factor's
backward error, and the iteration counts of plasma_dsposv against the oracle's.

Bounds: the FP32 factor's backward error ||A - L L^T|| / ||A|| does not depend
on the condition of A, so it is held to 1.5 times that of LAPACK's spotrf on
the same matrix, or to 3 u where that is more (LAPACK's is about u at small
orders).  Over 30 seeds panels by substitution reach 0.8 of this limit, panels
multiplied by the inverse of the whole tile 2 to 2.7 times it from order 48 on.
What is left is the inverse of a 16 x 16 diagonal block, whose rounding grows
with the block's condition: tiles of only a few such blocks get noise 1e-2,
with 1e-4 (blocks of condition 1e5) 5 u were measured at order 16.
The iteration count is the oracle's within 1; where it is beyond 10, or rests on
the accuracy of the solves with tile inverses, only convergence is asked for.
"""
import numpy as np
import pytest

import oracle as ora
import plasma_amd as pa
from tests import _util as U

pytestmark = pytest.mark.gpu

L, Up = pa.PlasmaLower, pa.PlasmaUpper


def _rbf(n, d, scale, noise, seed=0):
    X = np.random.default_rng(seed).random((n, d))
    if d == 1:
        X = np.sort(X, axis=0)
    D2 = sum((X[:, i, None] - X[None, :, i]) ** 2 for i in range(d))
    return np.asfortranarray(np.exp(-D2 / (2 * scale * scale)) +
                             noise * np.eye(n))


def _backward(A, F):
    F = F.astype(np.float64)
    return np.linalg.norm(A - F @ F.T) / np.linalg.norm(A)


@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,nb,noise", [
    (512, 128, 1e-4), (300, 128, 1e-4), (400, 112, 1e-4), (307, 100, 1e-4),
    (202, 65, 1e-4), (256, 64, 1e-4), (151, 48, 1e-4), (106, 33, 1e-2),
    (80, 16, 1e-2), (70, 7, 1e-2)])
def test_spotrf_backward_error(plasma, nb_guard, uplo, n, nb, noise):
    from scipy.linalg import lapack
    pa.set_param(pa.PlasmaNb, nb)
    S = _rbf(n, 1, 0.2, noise).astype(np.float32)
    A = S.astype(np.float64)
    ref, info = lapack.spotrf(S, lower=1)
    assert info == 0
    a = S.copy(order="F")
    assert pa.potrf(uplo, n, a, n, prec="s") == 0
    got = np.tril(a) if uplo == L else np.triu(a).T
    err = _backward(A, got)
    lim = max(1.5 * _backward(A, np.tril(ref)), 3 * U.EPS32)
    assert err <= lim, (err, lim)


@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,d,scale,noise,margin", [
    (512, 1, 0.2, 1e-3, 1),         # condition 2.3e5
    (512, 1, 0.2, 1e-4, 1),         # 2.3e6
    (512, 1, 0.2, 5e-5, 1),         # 4.6e6
    (512, 1, 0.2, 2e-5, None),      # 1.1e7
    (1024, 3, 0.5, 1e-4, 1),        # 4.7e6
    (2048, 2, 0.3, 1e-4, None),     # 7.2e6
])
def test_dsposv_iterations(plasma, nb_guard, uplo, n, d, scale, noise,
                           margin):
    nb, nrhs = 128, 3
    pa.set_param(pa.PlasmaNb, nb)
    A = _rbf(n, d, scale, noise)
    B = U.rhs(n, nrhs, seed=9)
    a, b = A.copy(order="F"), B.copy(order="F")
    X = np.zeros_like(b, order="F")
    info, it = pa.dsposv(uplo, n, nrhs, a, n, b, n, X, n)
    ora.set_blas(ora.MKL)
    _, ito, infoo = ora.dsposv(ora.LOWER if uplo == L else ora.UPPER, A, B,
                               nb)
    assert info == infoo == 0
    assert 0 <= it <= 30 and 0 <= ito <= 30, (it, ito)
    if margin is not None:
        assert abs(it - ito) <= margin, (it, ito)
    assert U.scaled_residual(A, X, B) < 10 * U.EPS64
