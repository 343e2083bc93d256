"""The resident evolver (one launch for many passes of a lattice of side <= 128, scalar_resident.hpp) and the
plane-chunk pass of ragged sides (scalar_flat.hpp).  The resident evolver is compared with the pass-by-pass
evolvers, which a context with pass timing on runs: the same operations in the same order, so fields, momenta,
background and constraint agree to the bit."""
import threading

import numpy as np
import pytest

from cosmolattice_amd.clmi import (CLMI_F32_BULK, CLMI_F64, CLMI_FLAG_NO_TILED, FLD_CS, FLD_S, FLD_U1, PI_CS, PI_S,
                                   PI_U1, PV_WEIGHTS, VV_WEIGHTS, Lattice, lphi4, lphi4U1)

pytestmark = pytest.mark.gpu


def model(kind):
    base = lphi4(100.0, n_fields=1 if kind == "1f" else 2, phi0_gev=5.6964e18, lam=1.0, pi0_program=-0.5)
    if kind == "terms":  # outside the compile-time potential
        base.terms = [(0.25, [4, 0]), (50.0, [2, 2]), (0.1, [0, 4]), (0.3, [2, 0])]
    return base


def start(spec, N, prec, expansion, seed=5):
    rng = np.random.default_rng(seed)
    lat = Lattice(spec, N, 0.4909, 0.005, prec, expansion=expansion)
    for k in (FLD_S, PI_S):
        for f in range(spec.n_scalars):
            lat.upload(k, f, 0, 0.3 * rng.standard_normal((N, N, N)) + (1.0 if k == FLD_S and f == 0 else 0.0))
    lat.set_background(aI=1.0, aSI=1.0, aIM=1.0, aDotI=0.7)
    lat.set_all_averages()
    return lat


def evolve(lat, scheme):
    """Calls of uneven length around the fewest passes the resident evolver takes, then the whole state."""
    for n in (6, 1, 5, 9):
        if scheme == "LF":
            if n == 6:
                lat.lf_init()
            lat.lf_evolve(n)
            if n == 5:
                lat.lf_sync()
        elif scheme.startswith("VV"):
            lat.vv_evolve(VV_WEIGHTS[scheme], n)
        else:
            lat.pv_evolve(PV_WEIGHTS[scheme], n)
    if scheme == "LF":
        lat.lf_sync()
    fields = [lat.download(k, f, 0) for k in (FLD_S, PI_S) for f in range(lat.spec.n_scalars)]
    return fields, lat.background(), lat.hubble_constraint()


@pytest.mark.parametrize("N", [32, 64, 100, 120, 128])
@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
@pytest.mark.parametrize("kind,scheme,expansion", [("2f", "LF", True), ("1f", "LF", True), ("terms", "LF", False),
                                                   ("2f", "VV4", True), ("1f", "VV2", True), ("2f", "PV4", True),
                                                   ("1f", "PV2", False)])
def test_resident_bit_identical_to_passes(gpu, N, prec, kind, scheme, expansion):
    print(f"case resident N={N} prec={prec} {kind} {scheme} expansion={expansion}", flush=True)
    spec = model(kind)
    res = []
    for timed in (False, True):
        lat = start(spec, N, prec, expansion)
        assert "k_scalar_resident" in lat.plan()
        if timed:
            lat.profile_enable(True, every=1 << 30)
        res.append(evolve(lat, scheme))
        lat.close()
    (fa, ba, ca), (fb, bb, cb) = res
    for a, b in zip(fa, fb):
        assert np.array_equal(a, b)
    assert ba == bb and ca == cb
    if expansion:
        assert ba["aI"] > 1.0


# chunk and group edges: one chunk per plane (24), chunks ending inside a row, full chunks (32, 96), the widest one-site
# and two-site lanes (62, 126), eight-plane tiles with a short last group (126), and sizes past the resident evolver
@pytest.mark.parametrize("N", [24, 32, 42, 62, 66, 96, 100, 126, 130, 250, 300])
@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
@pytest.mark.parametrize("kind,scheme", [("2f", "LF"), ("1f", "VV2"), ("terms", "PV2")])
def test_ragged_sides_bit_identical_to_one_site_per_thread(gpu, N, prec, kind, scheme):
    """The plane-chunk pass, pass by pass and (N <= 128) in the resident evolver, on a static background: fields
    and momenta equal the one-site-per-thread pass's to the bit; its sums differ in order only."""
    print(f"case ragged N={N} prec={prec} {kind} {scheme}", flush=True)
    spec = model(kind)
    rng = np.random.default_rng(N)
    ics = {(k, f): 0.3 * rng.standard_normal((N, N, N)) + (1.0 if (k, f) == (FLD_S, 0) else 0.0)
           for k in (FLD_S, PI_S) for f in range(spec.n_scalars)}
    res = []
    for how in ("one site", "passes", "default"):
        lat = Lattice(spec, N, 0.4909, 0.005, prec, expansion=False, flags=CLMI_FLAG_NO_TILED if how == "one site" else 0)
        plan = lat.plan()
        assert plan.split()[0] == ("k_scalar_pass" if how == "one site" else "k_scalar_flat")
        assert ("k_scalar_resident" in plan) == (how != "one site" and N <= 128)
        for (k, f), a in ics.items():
            lat.upload(k, f, 0, a)
        lat.set_background(aI=1.1, aSI=1.05, aIM=1.0)
        if how == "passes":
            lat.profile_enable(True, every=1 << 30)
        if scheme == "LF":
            lat.lf_init()
            lat.lf_evolve(6)
            lat.lf_sync()
        elif scheme == "VV2":
            lat.vv_evolve([1.0], 6)
        else:
            lat.pv_evolve([1.0], 4)
        res.append(([lat.download(k, f, 0) for k, f in ics], lat.averages()))
        lat.close()
    for fields, sums in res[1:]:
        for a, b in zip(res[0][0], fields):
            assert np.array_equal(a, b)
        for k in ("pi2S", "grad2S", "pot"):
            assert sums[k] == pytest.approx(res[0][1][k], rel=1e-13)
    assert res[1][1] == res[2][1]


U1_KINDS = [(FLD_CS, 0), (FLD_CS, 1), (PI_CS, 0), (PI_CS, 1)] + [(k, d) for k in (FLD_U1, PI_U1) for d in range(3)]


# tile edges: one short row tile (52, 62), two of 38 sites and a last tile of rows that is full (76), a short last tile of
# rows and x-chunk (90, 130)
@pytest.mark.parametrize("N", [52, 62, 76, 90, 130])
@pytest.mark.parametrize("prec", [CLMI_F64, CLMI_F32_BULK])
@pytest.mark.parametrize("scheme", ["LF", "VV2", "PV2"])
def test_ragged_u1_bit_identical_to_one_site_per_thread(gpu, N, prec, scheme):
    """The tiled charged-scalar + U(1) pass on a side that is no multiple of 64, static background: every array equals
    the one-site-per-thread pass's to the bit; its sums differ in order only."""
    print(f"case ragged u1 N={N} prec={prec} {scheme}", flush=True)
    spec = lphi4U1(10.0, phi0_gev=5.6964e18, lam=1.0, pi0_gev2=0.0)
    rng = np.random.default_rng(N)
    ics = {kc: 0.3 * rng.standard_normal((N, N, N)) for kc in U1_KINDS}
    res = []
    for flags, kernel in ((CLMI_FLAG_NO_TILED, "k_gauge_pass"), (0, "k_gauge_tiled")):
        lat = Lattice(spec, N, 0.4909, 0.005, prec, expansion=False, flags=flags)
        assert lat.plan().split()[0] == kernel
        for (k, c), a in ics.items():
            lat.upload(k, 0, c, a)
        lat.set_background(aI=1.1, aSI=1.05, aIM=1.0)
        if scheme == "LF":
            lat.lf_init()
            lat.lf_evolve(3)
            lat.lf_sync()
        elif scheme == "VV2":
            lat.vv_evolve([1.0], 2)
        else:
            lat.pv_evolve([1.0], 2)
        res.append(([lat.download(k, 0, c) for k, c in ics], lat.averages()))
        lat.close()
    for a, b in zip(res[0][0], res[1][0]):
        assert np.array_equal(a, b)
    for k in ("pi2CS", "grad2CS", "pot", "pi2U1", "B2U1"):
        assert res[1][1][k] == pytest.approx(res[0][1][k], rel=1e-13)


def test_resident_two_threads(gpu):
    """Two contexts driven by two host threads at once: each ends where it ends alone."""
    print("case resident two threads", flush=True)
    spec = model("2f")

    def run(seed, out):
        lat = start(spec, 128, CLMI_F32_BULK, True, seed)
        lat.lf_init()
        for _ in range(10):
            lat.lf_evolve(20)
        lat.lf_sync()
        out[seed] = [lat.download(k, f, 0) for k in (FLD_S, PI_S) for f in range(2)]
        lat.close()

    alone, together = {}, {}
    for seed in (1, 2):
        run(seed, alone)
    threads = [threading.Thread(target=run, args=(seed, together)) for seed in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for seed in (1, 2):
        for a, b in zip(alone[seed], together[seed]):
            assert np.array_equal(a, b)
