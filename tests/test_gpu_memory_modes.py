"""GPU: the memory mode of the full-row pass follows what of the state the last-level cache keeps (plans only; results do
not depend on it)."""
import pytest

from cosmolattice_amd.clmi import CLMI_F32_BULK, CLMI_F64, Lattice, lphi4
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


# state in both buffers: 50 and 226 MB (in the cache), 340, 403 and 453 MB (one buffer in it), 805 MB (one buffer up to twice
# the cache), 6.4 GB
@pytest.mark.parametrize("N,prec,nf,mode", [(128, CLMI_F32_BULK, 1, 0), (192, CLMI_F64, 1, 0), (192, CLMI_F32_BULK, 2, 1),
                                            (256, CLMI_F32_BULK, 1, 1), (192, CLMI_F64, 2, 1),
                                            (256, CLMI_F32_BULK, 2, 15), (512, CLMI_F32_BULK, 2, 1)])
def test_default_memory_mode(gpu, N, prec, nf, mode):
    say(f"case memory mode N={N} prec={prec} nf={nf}")
    spec = lphi4(100.0, n_fields=nf, phi0_gev=5.6964e18, lam=1.0, pi0_program=-0.5)
    lat = Lattice(spec, N, 0.4909, 0.005, prec)
    assert f" MM={mode} " in lat.plan().splitlines()[0]
    lat.close()
