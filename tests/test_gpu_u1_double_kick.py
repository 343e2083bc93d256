"""Velocity Verlet of a charged scalar with and without U(1): two kicks in one tiled pass against one pass each."""
import numpy as np
import pytest

from cosmolattice_amd.clmi import (CLMI_F32_BULK, CLMI_F64, CLMI_FLAG_NO_DOUBLE_KICK, FLD_CS, FLD_S, FLD_U1, PI_CS,
                                   PI_S, PI_U1, VV_WEIGHTS, Lattice, lphi4, lphi4U1)

pytestmark = pytest.mark.gpu


# ragged tiles (52, the smallest; 90, short last tiles of rows, sites and x-chunk), full tiles that stay in the last-level
# cache or not (64; 128 in FP64); a composition with a kick of weight zero, which no pass may take as a second kick
@pytest.mark.parametrize("N,weights", [(52, "VV2"), (64, "VV4"), (90, "VV4"), (128, "VV2"), (64, "zero")])
@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
@pytest.mark.parametrize("u1", [True, False])
@pytest.mark.parametrize("expansion", [True, False])
def test_double_kick_bit_identical_to_two_passes(gpu, N, weights, prec, u1, expansion):
    print(f"case u1 double kick N={N} {weights} prec={prec} u1={u1} expansion={expansion}", flush=True)
    spec = lphi4U1(10.0, phi0_gev=5.6964e18, lam=1.0, pi0_gev2=0.0)
    kinds = [(FLD_CS, 0), (FLD_CS, 1), (PI_CS, 0), (PI_CS, 1)]
    if u1:
        kinds += [(k, d) for k in (FLD_U1, PI_U1) for d in range(3)]
    else:
        spec.n_u1 = 0
    ws = [0.75, 0.0, -0.5] if weights == "zero" else VV_WEIGHTS[weights]
    rng = np.random.default_rng(N)
    ics = {kc: 0.3 * rng.standard_normal((N, N, N)) for kc in kinds}
    res = []
    for flags in (CLMI_FLAG_NO_DOUBLE_KICK, 0):
        lat = Lattice(spec, N, 0.4909, 0.005, prec, expansion=expansion, flags=flags)
        assert lat.plan().split()[0] == "k_gauge_tiled"
        for (k, c), a in ics.items():
            lat.upload(k, 0, c, a)
        lat.set_background(aI=1.1, aSI=1.05, aIM=1.0, aDotI=0.2, aDotSI=0.2)
        lat.set_all_averages()
        lat.vv_evolve(ws, 3)
        res.append(([lat.download(k, 0, c) for k, c in kinds], lat.background(), lat.averages()))
        lat.close()
    for a, b in zip(res[0][0], res[1][0]):
        assert np.array_equal(a, b)
    assert res[0][1:] == res[1][1:]


@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
def test_scalar_weight_zero_takes_two_passes(gpu, prec):
    """The averages after a kick of weight zero are those of the momenta, not of a second sum that no pass formed."""
    print(f"case scalar weight zero prec={prec}", flush=True)
    spec = lphi4(100.0, phi0_gev=5.6964e18, lam=1.0, pi0_program=-0.5)
    rng = np.random.default_rng(5)
    ics = {(k, f): 0.3 * rng.standard_normal((64, 64, 64)) for k in (FLD_S, PI_S) for f in range(2)}
    res = []
    for flags in (CLMI_FLAG_NO_DOUBLE_KICK, 0):
        lat = Lattice(spec, 64, 0.4909, 0.005, prec, flags=flags)
        for (k, f), a in ics.items():
            lat.upload(k, f, 0, a)
        lat.set_background(aI=1.1, aSI=1.05, aIM=1.0, aDotI=0.2, aDotSI=0.2)
        lat.set_all_averages()
        lat.vv_evolve([0.75, 0.0, -0.5], 3)
        res.append(([lat.download(k, f, 0) for k, f in ics], lat.background()))
        lat.close()
    for a, b in zip(res[0][0], res[1][0]):
        assert np.array_equal(a, b)
    assert res[0][1] == res[1][1]
