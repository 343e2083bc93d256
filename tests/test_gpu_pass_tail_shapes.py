"""GPU: the background update in the last workgroup of full-row passes whose workgroups are smaller (256 threads, each
standing for two of the update's 512 summing threads) or larger (1024) than the default 512, against the update launch of
its own, which passes timed one by one keep: bit for bit."""
import numpy as np
import pytest

from cosmolattice_amd.clmi import (CLMI_F32_BULK, CLMI_F64, CLMI_FLAG_MEMMODE, CLMI_FLAG_SHAPE_ALT, CLMI_FLAG_SHAPE_TY4,
                                   FLD_S, PI_S, VV_WEIGHTS, Lattice, lphi4)
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
@pytest.mark.parametrize("flags,shape", [(CLMI_FLAG_SHAPE_ALT | CLMI_FLAG_SHAPE_TY4, "VZ=4 WPR=1 TY=4"),
                                         (CLMI_FLAG_MEMMODE(1), "VZ=2 WPR=2 TY=8")])
@pytest.mark.parametrize("scheme", ["LF", "VV2"])
def test_update_in_pass_of_other_workgroups(gpu, prec, flags, shape, scheme):
    say(f"case pass tail shapes prec={prec} {shape} {scheme}")
    N = 256
    spec = lphi4(100.0, phi0_gev=5.6964e18, lam=1.0, pi0_program=-0.5)
    rng = np.random.default_rng(7)
    ics = {(k, f): 0.3 * rng.standard_normal((N, N, N)) + (1.0 if (k, f) == (FLD_S, 0) else 0.0)
           for k in (FLD_S, PI_S) for f in range(2)}
    res = []
    for every in (1 << 30, 1):  # 1: every drift + kick pass is timed by itself, with its update's launch after it
        lat = Lattice(spec, N, 0.4909, 0.005, prec, flags=flags)
        assert lat.plan().startswith("k_scalar_rows " + shape)
        for (k, f), a in ics.items():
            lat.upload(k, f, 0, a)
        lat.set_background(aI=1.0, aSI=1.0, aIM=1.0, aDotI=0.7)
        lat.set_all_averages()
        lat.profile_enable(True, every=every)
        if scheme == "LF":
            lat.lf_init()
            lat.lf_evolve(5)
            lat.lf_sync()
        else:
            lat.vv_evolve(VV_WEIGHTS[scheme], 3)
        res.append(([lat.download(k, f, 0) for k, f in sorted(ics)], lat.background()))
        lat.close()
    assert res[0][1] == res[1][1] and res[0][1]["aI"] > 1.0
    for a, b in zip(res[0][0], res[1][0]):
        assert np.array_equal(a, b)
