"""GPU: the gate of the resident evolver.  Its workgroups evolve nothing until all have started; where they cannot, the
gate closes, the state passes through unchanged, and the context's next call takes the passes one by one, as all later
ones do, with the same bits.  CLMI_FLAG_REFUSE_RESIDENT keeps the gate shut from the host."""
import numpy as np
import pytest

from cosmolattice_amd.clmi import (CLMI_F32_BULK, CLMI_F64, CLMI_FLAG_REFUSE_RESIDENT, FLD_S, PI_S, PV_WEIGHTS,
                                   VV_WEIGHTS, Ensemble, Lattice, lphi4)
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


def start(N, prec, expansion, flags):
    spec = lphi4(100.0, phi0_gev=5.6964e18, lam=1.0, pi0_program=-0.5)
    rng = np.random.default_rng(N)
    lat = Lattice(spec, N, 0.4909, 0.005, prec, expansion=expansion, flags=flags)
    for k in (FLD_S, PI_S):
        for f in range(2):
            lat.upload(k, f, 0, 0.3 * rng.standard_normal((N, N, N)) + (1.0 if (k, f) == (FLD_S, 0) else 0.0))
    lat.set_background(aI=1.0, aSI=1.0, aIM=1.0, aDotI=0.7)
    lat.set_all_averages()
    lat.lf_init()
    return lat


def state(lat):
    return [lat.download(k, f, 0) for k in (FLD_S, PI_S) for f in range(2)], lat.background()


# two, four and eight planes a tile, full and ragged ones
@pytest.mark.parametrize("N", [32, 64, 100, 128])
@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
@pytest.mark.parametrize("scheme,expansion", [("LF", True), ("LF", False), ("VV2", True), ("PV4", True)])
def test_closed_gate_leaves_the_passes(gpu, N, prec, scheme, expansion):
    say(f"case gate N={N} prec={prec} {scheme} expansion={expansion}")
    res = []
    for flags in (0, CLMI_FLAG_REFUSE_RESIDENT):
        lat = start(N, prec, expansion, flags)
        assert "k_scalar_resident" in lat.plan()
        for n in (7, 5, 9):  # the first of them meets the gate; the whole state must be what its passes leave
            if scheme == "LF":
                lat.lf_evolve(n)
            elif scheme == "VV2":
                lat.vv_evolve(VV_WEIGHTS[scheme], n)
            else:
                lat.pv_evolve(PV_WEIGHTS[scheme], n)
            # an open gate keeps the evolver in use, a closed one ends it (at the context's next call)
            lat.synchronize()
            assert ("k_scalar_resident" in lat.plan()) == (flags == 0)
        if scheme == "LF":
            lat.lf_sync()
        res.append(state(lat))
        lat.close()
    assert res[0][1] == res[1][1]
    for a, b in zip(res[0][0], res[1][0]):
        assert np.array_equal(a, b)


def test_ensemble_of_members_with_a_closed_gate(gpu):
    say("case gate ensemble")
    res = []
    for flags in (0, CLMI_FLAG_REFUSE_RESIDENT):
        lats = [start(N, CLMI_F64, True, flags) for N in (64, 128)]
        for lat in lats:
            lat.lf_evolve(6)
        ens = Ensemble(lats)
        ens.lf_evolve(5)
        for lat in lats:
            lat.lf_sync()
        res.append([state(lat) for lat in lats])
        ens.close()
        for lat in lats:
            lat.close()
    for (fa, ba), (fb, bb) in zip(*res):
        assert ba == bb
        for a, b in zip(fa, fb):
            assert np.array_equal(a, b)
