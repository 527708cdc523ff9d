"""GPU tests of the batched solver's classes of orders (up to 128, 256, 512):
orders around the 16-row blocks and the class limits, 1 to 16 right-hand
sides (17 takes the other kernel), both storages and precisions, offsets that
leave systems without 16-byte alignment, and a failing system between others
whose right-hand sides must stay as they were.

Bounds: factor 4 sqrt(n) u relative, scaled residual 10 u (u = 2^-53, 2^-24), on
matrices G G^T / n + I.
"""
import numpy as np
import pytest

import plasma_amd as pa
from tests import _util as U

pytestmark = pytest.mark.gpu

L, Up = pa.PlasmaLower, pa.PlasmaUpper
ORDERS = [1, 15, 16, 17, 33, 63, 64, 127, 128, 129, 200, 255, 256, 257, 400,
          511, 512, 0, 7]


def _run(prec, uplo, mats, rhs, nrhs, pad):
    import torch
    dt = np.float64 if prec == "d" else np.float32
    n = np.array([len(m) for m in mats], dtype=np.int32)
    aoff = np.zeros(len(mats), dtype=np.uint64)
    boff = np.zeros(len(mats), dtype=np.uint64)
    pa_, pb = pad, pad
    for i, k in enumerate(n):
        aoff[i], boff[i] = pa_, pb
        pa_ += int(k) * int(k) + pad
        pb += int(k) * nrhs + pad
    A = np.full(pa_ + 1, 9.0, dtype=dt)
    B = np.full(pb + 1, 9.0, dtype=dt)
    for i, k in enumerate(n):
        A[int(aoff[i]):int(aoff[i]) + k * k] = mats[i].ravel(order="F")
        B[int(boff[i]):int(boff[i]) + k * nrhs] = rhs[i].ravel(order="F")
    dA, dB = torch.from_numpy(A.copy()).cuda(), torch.from_numpy(B.copy()).cuda()
    info = np.full(len(mats), -7, dtype=np.int32)
    torch.cuda.synchronize()
    rc = getattr(pa.load(), "plasma_%sposv_vbatched" % prec)(
        uplo, len(mats), n.ctypes.data, dA.data_ptr(), aoff.ctypes.data, nrhs,
        dB.data_ptr(), boff.ctypes.data, info.ctypes.data)
    assert rc == 0
    a, b = dA.cpu().numpy(), dB.cpu().numpy()
    used = np.zeros(len(A), dtype=bool)
    outA, outB = [], []
    for i, k in enumerate(n):
        o = int(aoff[i])
        used[o:o + k * k] = True
        outA.append(a[o:o + k * k].reshape(k, k, order="F"))
        o = int(boff[i])
        outB.append(b[o:o + k * nrhs].reshape(k, nrhs, order="F"))
    assert np.all(a[~used] == 9.0)
    return info, outA, outB


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("nrhs,pad", [(1, 0), (3, 1), (16, 3), (17, 0)])
def test_classes(plasma, prec, uplo, nrhs, pad):
    dt = np.float64 if prec == "d" else np.float32
    eps = U.EPS64 if prec == "d" else U.EPS32
    mats = [U.ggt_spd(k, seed=k).astype(dt) if k else np.zeros((0, 0), dt)
            for k in ORDERS]
    rhs = [U.rhs(k, nrhs, seed=k + 1).astype(dt) for k in ORDERS]
    bad = ORDERS.index(200)
    mats[bad][150, 150] = -1.0
    info, F, X = _run(prec, uplo, mats, rhs, nrhs, pad)
    for i, k in enumerate(ORDERS):
        if i == bad:
            assert info[i] == 151
            assert np.array_equal(X[i], rhs[i])
            continue
        assert info[i] == 0
        if k == 0:
            continue
        M = mats[i].astype(np.float64)
        ref = np.linalg.cholesky(M)
        got = np.tril(F[i]) if uplo == L else np.triu(F[i]).T
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert err <= 4 * np.sqrt(k) * eps, (k, err)
        keep = np.triu(mats[i], 1) if uplo == L else np.tril(mats[i], -1)
        other = np.triu(F[i], 1) if uplo == L else np.tril(F[i], -1)
        assert np.array_equal(other, keep), k
        res = U.scaled_residual(M, X[i].astype(np.float64),
                                rhs[i].astype(np.float64))
        assert res <= 10 * eps, (k, res)
