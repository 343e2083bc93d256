"""The background update in the last workgroup of a full-row or plane-chunk pass (pass_tail.hpp) against the update
launch of its own, which passes that are timed one by one keep: the same sums in the same order and the same operations,
so fields, momenta and background agree to the bit."""
import numpy as np
import pytest

from cosmolattice_amd.clmi import (CLMI_F32_BULK, CLMI_F64, FLD_S, PI_S, PV_WEIGHTS, VV_WEIGHTS, Lattice, lphi4)

pytestmark = pytest.mark.gpu


# fewer rows than the update's 512 summing threads (24, 32), one and several a thread; workgroups of 128 to 1024 threads
@pytest.mark.parametrize("N", [24, 32, 64, 100, 128, 192, 256, 300])
@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
@pytest.mark.parametrize("nf,scheme", [(2, "LF"), (1, "VV2"), (2, "PV2")])
def test_update_in_pass_bit_identical_to_its_own_launch(gpu, N, prec, nf, scheme):
    print(f"case pass tail N={N} prec={prec} {nf}f {scheme}", flush=True)
    spec = lphi4(100.0, n_fields=nf, phi0_gev=5.6964e18, lam=1.0, pi0_program=-0.5)
    rng = np.random.default_rng(N)
    ics = {(k, f): 0.3 * rng.standard_normal((N, N, N)) + (1.0 if (k, f) == (FLD_S, 0) else 0.0)
           for k in (FLD_S, PI_S) for f in range(nf)}
    res = []
    for every in (1 << 30, 1):
        lat = Lattice(spec, N, 0.4909, 0.005, prec)
        for (k, f), a in ics.items():
            lat.upload(k, f, 0, a)
        lat.set_background(aI=1.0, aSI=1.0, aIM=1.0, aDotI=0.7)
        lat.set_all_averages()
        lat.profile_enable(True, every=every)
        if scheme == "LF":
            lat.lf_init()
            lat.lf_evolve(7)
            lat.lf_sync()
        elif scheme == "VV2":
            lat.vv_evolve(VV_WEIGHTS[scheme], 4)
        else:
            lat.pv_evolve(PV_WEIGHTS[scheme], 4)
        res.append(([lat.download(k, f, 0) for k, f in sorted(ics)], lat.background()))
        lat.close()
    (fa, ba), (fb, bb) = res
    assert ba == bb and ba["aI"] > 1.0
    for a, b in zip(fa, fb):
        assert np.array_equal(a, b)
