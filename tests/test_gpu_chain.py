"""GPU tests of the small-block panel solve and trailing update: tile sizes
that are no multiple of the blocks (32, 64) or of the K chunk (8 in FP64, 16
in FP32), K shorter than the ring of chunks, several update depths and
lookaheads, both storages and precisions.

Bound: the factor's relative error stays within 4 sqrt(n) u for these
well-conditioned matrices (u = 2^-53, 2^-24).
"""
import numpy as np
import pytest

import plasma_amd as pa
from tests import _util as U

pytestmark = pytest.mark.gpu

L, Up = pa.PlasmaLower, pa.PlasmaUpper


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,nb,depth,la", [
    (67, 5, 1, 0), (130, 20, 3, 1), (301, 36, 2, 1), (515, 100, 4, 0),
    (700, 65, 1, 1), (640, 128, 3, 2), (1290, 128, 4, 1), (1100, 200, 2, 1)])
def test_factor(plasma, nb_guard, prec, uplo, n, nb, depth, la):
    pa.set_param(pa.PlasmaNb, nb)
    pa.set_param(pa.PlasmaUpdateDepth, depth)
    pa.set_param(pa.PlasmaLookahead, la)
    dt = np.float64 if prec == "d" else np.float32
    eps = U.EPS64 if prec == "d" else U.EPS32
    A = U.ggt_spd(n, seed=n).astype(dt)
    lda = n + 1
    a = np.zeros((lda, n), dtype=dt, order="F")
    a[:n] = A
    assert pa.potrf(uplo, n, a, lda, prec=prec) == 0
    ref = np.linalg.cholesky(A.astype(np.float64))
    got = np.tril(a[:n]) if uplo == L else np.triu(a[:n]).T
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= 4 * np.sqrt(n) * eps, err
    keep = np.triu(A, 1) if uplo == L else np.tril(A, -1)
    other = np.triu(a[:n], 1) if uplo == L else np.tril(a[:n], -1)
    assert np.array_equal(other, keep)
