"""GPU tests of pivots below the smallest normal number: a positive pivot is
accepted whatever its size (LAPACK takes its square root), so the factor and
the solution of a diagonal matrix of powers of four are exact.  All precisions,
tiles of one and of several 16-column panels, and the batched solver.
"""
import numpy as np
import pytest

import plasma_amd as pa

pytestmark = pytest.mark.gpu

L, Up = pa.PlasmaLower, pa.PlasmaUpper
DT = {"d": np.float64, "s": np.float32, "z": np.complex128,
      "c": np.complex64}
# exponent of the small pivots, of their right-hand sides
EXP = {"d": (-1040, -540), "z": (-1040, -540), "s": (-140, -100),
       "c": (-140, -100)}


def _system(prec, n):
    e, f = EXP[prec]
    small = np.arange(n) % 3 == (n - 1) % 3         # the last one among them
    diag = np.where(small, np.ldexp(1.0, e), 4.0)
    root = np.where(small, np.ldexp(1.0, e // 2), 2.0)
    b = np.where(small, np.ldexp(1.0, f), 1.0)
    x = np.where(small, np.ldexp(1.0, f - e), 0.25)
    dt = DT[prec]
    assert np.all(diag.astype(dt) == diag)
    return (np.asfortranarray(np.diag(diag).astype(dt)),
            np.diag(root).astype(dt), b.astype(dt), x.astype(dt))


@pytest.mark.parametrize("prec", ["d", "s", "z", "c"])
@pytest.mark.parametrize("uplo", [L, Up])
@pytest.mark.parametrize("n,nb", [(1, 128), (16, 128), (40, 128), (128, 128),
                                  (100, 40)])
def test_posv(plasma, nb_guard, prec, uplo, n, nb):
    pa.set_param(pa.PlasmaNb, nb)
    A, F, b, x = _system(prec, n)
    b = np.asfortranarray(b[:, None])
    assert pa.posv(uplo, n, 1, A, n, b, n, prec=prec) == 0
    assert np.array_equal(A, F)
    assert np.array_equal(b[:, 0], x)


@pytest.mark.parametrize("prec", ["d", "s"])
@pytest.mark.parametrize("uplo", [L, Up])
def test_batched(plasma, prec, uplo):
    orders = [1, 16, 40, 128, 130, 300]
    systems = [_system(prec, n) for n in orders]
    n = np.array(orders, dtype=np.int32)
    aoff = np.concatenate([[0], np.cumsum(n * n)[:-1]]).astype(np.uint64)
    boff = np.concatenate([[0], np.cumsum(n)[:-1]]).astype(np.uint64)
    A = np.concatenate([s[0].ravel() for s in systems])
    B = np.concatenate([s[2] for s in systems])
    import torch
    dA, dB = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    info = np.full(len(n), -7, dtype=np.int32)
    torch.cuda.synchronize()
    assert getattr(pa.load(), "plasma_%sposv_vbatched" % prec)(
        uplo, len(n), n.ctypes.data, dA.data_ptr(), aoff.ctypes.data, 1,
        dB.data_ptr(), boff.ctypes.data, info.ctypes.data) == 0
    assert not info.any()
    a, b = dA.cpu().numpy(), dB.cpu().numpy()
    for s, k, oa, ob in zip(systems, orders, aoff.astype(int),
                            boff.astype(int)):
        assert np.array_equal(a[oa:oa + k * k].reshape(k, k), s[1])
        assert np.array_equal(b[ob:ob + k], s[3])
