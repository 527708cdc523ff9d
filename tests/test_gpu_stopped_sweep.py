"""GPU test of the one-launch triangular sweeps when the sequence's status
word is set: every workgroup must still publish its block row, because others
that saw the word clear may be waiting for it.  The word is set before the
launch here, so no workgroup waits; after it every flag of every group that
holds right-hand sides is set.
"""
import ctypes

import numpy as np
import pytest

import plasma_amd as pa

pytestmark = pytest.mark.gpu

PREC = {"d": (pa.PlasmaRealDouble, np.float64, 16, "flow"),
        "s": (pa.PlasmaRealFloat, np.float32, 16, "flow"),
        "z": (pa.PlasmaComplexDouble, np.complex128, 8, "zflow"),
        "c": (pa.PlasmaComplexFloat, np.complex64, 8, "zflow")}


@pytest.mark.parametrize("prec", ["d", "s", "z", "c"])
@pytest.mark.parametrize("backward", [0, 1])
def test_all_flags_set(plasma, nb_guard, prec, backward):
    import torch
    kind, dt, cols, name = PREC[prec]
    n, nb, nrhs = 200, 64, 2 * cols + 3
    lib = pa.load()
    A, B = pa.plasma_desc_t(), pa.plasma_desc_t()
    assert lib.plasma_desc_triangular_create(
        kind, pa.PlasmaLower, nb, nb, n, n, 0, 0, n, n,
        ctypes.byref(A)) == 0
    assert lib.plasma_desc_general_create(
        kind, nb, nb, n, nrhs, 0, 0, n, nrhs, ctypes.byref(B)) == 0
    launch = getattr(lib, "plasma_kern_%s_sweep" % name)
    ints = getattr(lib, "plasma_%s_sweep_ints" % name)
    launch.restype, ints.restype = ctypes.c_int, ctypes.c_size_t
    launch.argtypes = [ctypes.c_int, ctypes.c_int, pa.plasma_desc_t,
                       pa.plasma_desc_t] + [ctypes.c_void_p] * 4
    ints.argtypes = [pa.plasma_desc_t]
    size = ints(B)
    inv = torch.zeros(A.mt * nb * nb, dtype=torch.from_numpy(
        np.zeros(1, dtype=dt)).dtype, device="cuda")
    sync = torch.zeros(size, dtype=torch.int32, device="cuda")
    status = torch.full((1,), 7, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    assert launch(pa.PlasmaLower, backward, A, B, inv.data_ptr(),
                  sync.data_ptr(), status.data_ptr(), None) == 0
    torch.cuda.synchronize()
    got = sync.cpu().numpy()
    lib.plasma_desc_destroy(ctypes.byref(A))
    lib.plasma_desc_destroy(ctypes.byref(B))
    groups = (nb + cols - 1) // cols * B.nt
    used = (nrhs + cols - 1) // cols
    assert got[0] == B.mt * groups                  # one ticket each
    flags = got[1:1 + groups * B.mt].reshape(groups, B.mt)
    assert np.all(flags[:used] == 1), flags
