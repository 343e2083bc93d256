"""Downloads of 32 MB and more into pageable memory go through a page-locked buffer by several threads (host_read); into
page-locked memory, and below 32 MB, they are one copy.  What is written is the same: the array's doubles, to the last
partial chunk, and nothing beyond it."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from cosmolattice_amd.clmi import CLMI_F32_BULK, CLMI_F64, FLD_S, PI_S, Lattice, lphi4

pytestmark = pytest.mark.gpu


def roundtrip(N, prec, pinned, shift):
    """Uploads random fields, downloads them to `shift` doubles past the start of a guarded buffer."""
    lat = Lattice(lphi4(100.0, n_fields=2), N, 0.4909, 0.005, prec)
    rng = np.random.default_rng(N)
    for kind in (FLD_S, PI_S):
        for f in range(2):
            # FP32 pairs and singles hold these exactly
            a = rng.standard_normal(N ** 3).astype(np.float32).astype(np.float64)
            lat.upload(kind, f, 0, a.reshape(N, N, N))
            buf = torch.full((N ** 3 + 8,), -7.0, dtype=torch.float64, pin_memory=pinned).numpy()
            out = buf[shift:]
            rc = lat.lib.clmi_download_field(lat.handle, kind, f, 0, out.ctypes.data_as(ctypes.POINTER(ctypes.c_double)))
            assert rc == 0
            assert np.array_equal(out[:N ** 3], a)
            assert np.all(buf[:shift] == -7.0) and np.all(out[N ** 3:] == -7.0)
    lat.close()


# the last size below 32 MB, the first above (a partial last chunk), whole chunks
@pytest.mark.parametrize("N", [160, 162, 192])
@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
@pytest.mark.parametrize("pinned,shift", [(False, 0), (False, 3), (True, 1)])
def test_download_is_exact(gpu, N, prec, pinned, shift):
    print(f"case host read N={N} prec={prec} pinned={pinned} shift={shift}", flush=True)
    roundtrip(N, prec, pinned, shift)


def test_downloads_of_two_threads(gpu):
    errs = []

    def run(N):
        try:
            roundtrip(N, CLMI_F64, False, 0)
        except BaseException as e:  # noqa: BLE001
            errs.append(e)

    th = [threading.Thread(target=run, args=(N,)) for N in (170, 192)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errs
