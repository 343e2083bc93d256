"""GPU: the resident evolver exchanges through the buffers that are not current and takes no memory of the lattice's size
for itself, whose release would cost a short-lived context more than the evolver gains it."""
import numpy as np
import pytest

from cosmolattice_amd.clmi import (CLMI_F32_BULK, CLMI_F64, FLD_S, PI_S, PV_WEIGHTS, VV_WEIGHTS, Lattice, lphi4)
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
@pytest.mark.parametrize("nf", [1, 2])
def test_first_resident_call_takes_little_memory(gpu, prec, nf):
    import torch

    say(f"case resident memory prec={prec} nf={nf}")
    N = 128
    spec = lphi4(100.0, n_fields=nf, phi0_gev=5.6964e18, lam=1.0, pi0_program=-0.5)
    # the process's first cooperative launch makes the runtime allocate its queue for them
    first = Lattice(spec, 32, 0.4909, 0.005, prec)
    first.lf_init()
    first.lf_evolve(8)
    first.synchronize()
    lat = Lattice(spec, N, 0.4909, 0.005, prec)
    for k in (FLD_S, PI_S):
        for f in range(nf):
            lat.upload(k, f, 0, 0.3 * np.random.default_rng(f).standard_normal((N, N, N)))
    lat.set_background(aI=1.0, aSI=1.0, aIM=1.0, aDotI=0.7)
    lat.set_all_averages()
    lat.lf_init()
    lat.lf_evolve(1)
    lat.synchronize()
    free = torch.cuda.mem_get_info()[0]
    lat.lf_evolve(8)
    lat.lf_sync()
    lat.vv_evolve(VV_WEIGHTS["VV2"], 8)
    lat.pv_evolve(PV_WEIGHTS["PV2"], 8)
    assert "k_scalar_resident" in lat.plan()
    # a momentum array is 8 or 16 MiB; a few small allocations share at most two blocks of 2 MiB
    assert free - torch.cuda.mem_get_info()[0] < 5 << 20
    lat.close()
    first.close()
