"""GPU: the autotuners time the plan that runs now, whatever its x-chunk, so that a default is only replaced by a chunk
that was faster; results do not depend on it."""
import re

import numpy as np
import pytest

from cosmolattice_amd.clmi import (CLMI_F32_BULK, CLMI_F64, FLD_CS, FLD_S, FLD_U1, PI_CS, PI_S, PI_U1, Ensemble,
                                   Lattice, lphi4, lphi4U1)
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

U1_KINDS = [(k, c) for k in (FLD_CS, PI_CS) for c in (0, 1)] + [(k, d) for k in (FLD_U1, PI_U1) for d in range(3)]


# default x-chunks that are no power of two (90, 100: 12), one row group (52), and sides of several row groups a chunk
@pytest.mark.parametrize("N", [52, 90, 100, 130])
@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
def test_autotune_times_the_ragged_u1_default(gpu, N, prec):
    say(f"case autotune ragged u1 N={N} prec={prec}")
    spec = lphi4U1(10.0, phi0_gev=5.6964e18, lam=1.0, pi0_gev2=0.0)
    rng = np.random.default_rng(N)
    ics = {kc: 0.3 * rng.standard_normal((N, N, N)) for kc in U1_KINDS}
    res = []
    for tune in (False, True):
        lat = Lattice(spec, N, 0.4909, 0.005, prec, expansion=False)
        for (k, c), a in ics.items():
            lat.upload(k, 0, c, a)
        lat.set_background(aI=1.1, aSI=1.05, aIM=1.0)
        if tune:
            xc = int(re.search(r"k_gauge_tiled TY=4 XC=(\d+)", lat.plan()).group(1))
            rep = lat.autotune(2)
            say(f"default XC={xc}\n{rep}")
            timed = {int(x): float(us) for x, us in re.findall(r"gauge XC=(\d+) ([\d.]+)", rep)}
            chosen = int(re.search(r"k_gauge_tiled TY=4 XC=(\d+)", rep).group(1))
            assert xc in timed and chosen in timed
            assert chosen == xc or timed[chosen] < timed[xc]
        lat.lf_init()
        lat.lf_evolve(2)
        lat.lf_sync()
        res.append(([lat.download(k, 0, c) for k, c in ics], lat.averages()))
        lat.close()
    assert res[0][1] == res[1][1]
    for a, b in zip(res[0][0], res[1][0]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
def test_ensemble_autotune_times_the_members_plans(gpu, prec):
    """Each size class's current x-chunk (24 at 192^3) is among those timed, and the one chosen was timed fastest."""
    say(f"case ensemble autotune prec={prec}")
    spec = lphi4(100.0, phi0_gev=5.6964e18, lam=1.0, pi0_program=-0.5)
    rng = np.random.default_rng(1)
    members = []
    for N in (64, 64, 128, 192):
        lat = Lattice(spec, N, 0.4909, 0.005, prec, expansion=False)
        for k in (FLD_S, PI_S):
            for f in range(2):
                lat.upload(k, f, 0, 0.3 * rng.standard_normal((N, N, N)))
        members.append(lat)
    chunks = {N: re.search(r" XC=(\d+)", lat.plan()).group(1) for N, lat in zip((64, 64, 128, 192), members)}
    ens = Ensemble(members)
    rep = ens.autotune(2)
    say(f"defaults {chunks}\n{rep}")
    for line, N in zip(rep.strip().splitlines(), (64, 128, 192)):
        timed = {x: float(us) for x, us in re.findall(r"XC=(\d+):([\d.]+)", line)}
        chosen = line.split("-> XC=")[1]
        assert chunks[N] in timed
        assert timed[chosen] == min(timed.values())
    ens.close()
    for lat in members:
        lat.close()
