"""Spectra of 64^3, 128^3 and 256^3, whose x transform runs inside the binning kernel, against numpy's transform binned with
the same formula.  White noise fills every bin, so each sum of >= 1 positive terms carries the transform's relative error,
about log2(N^3) roundings of 1.1e-16 a mode: 1e-12 leaves a factor of more than 100."""
import numpy as np
import pytest

from cosmolattice_amd.clmi import CLMI_F32_BULK, CLMI_F64, FLD_S, PI_S, Lattice, lphi4

pytestmark = pytest.mark.gpu


def binned(a, dk, nb, npow):
    N = a.shape[0]
    f2 = np.abs(np.fft.rfftn(a)) ** 2
    n = np.fft.fftfreq(N, 1.0 / N)
    kz = np.arange(N // 2 + 1)
    n2 = n[:, None, None] ** 2 + n[None, :, None] ** 2 + kz[None, None, :] ** 2
    w = np.where((kz == 0) | (2 * kz == N), 1.0, 2.0)[None, None, :]
    b = np.minimum(np.floor(np.sqrt(n2) / dk + 0.5).astype(int), nb - 1)
    return np.bincount(b.ravel(), (w * f2 * np.sqrt(n2) ** npow).ravel(), nb)


# dk = 2.5 joins many modes a bin, 0.3 leaves empty bins (and at 256^3 more than fit the fused kernel's histograms)
@pytest.mark.parametrize("N", [64, 128, 256])
@pytest.mark.parametrize("prec,kind", [(CLMI_F64, FLD_S), (CLMI_F32_BULK, PI_S)])
@pytest.mark.parametrize("dk,npow", [(1.0, 0), (2.5, 1), (0.3, 3)])
def test_spectrum_matches_numpy(gpu, N, prec, kind, dk, npow):
    print(f"case spectrum N={N} prec={prec} kind={kind} dk={dk} npow={npow}", flush=True)
    lat = Lattice(lphi4(100.0, n_fields=2), N, 0.4909, 0.005, prec)
    a = np.random.default_rng(N).standard_normal((N, N, N)).astype(np.float32).astype(np.float64)
    lat.upload(kind, 1, 0, a)
    for _ in range(2):
        got = lat.spectrum_bins(kind, 1, 0, dk=dk, npow=npow)[0]
        ref = binned(a, dk, len(got), npow)
        assert np.all(np.abs(got - ref) <= 1e-12 * ref)
    lat.close()
