"""GPU: two processes on one card.  The runtime gives cooperative launches to one process at a time; the other's are refused
(hipErrorIllegalState), and its lattices take their passes one by one, with the same bits."""
import hashlib
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parents[1]


def evolve():
    from cosmolattice_amd.clmi import CLMI_F64, FLD_S, PI_S, VV_WEIGHTS, Lattice, lphi4

    N = 64
    lat = Lattice(lphi4(100.0, phi0_gev=5.6964e18, lam=1.0, pi0_program=-0.5), N, 0.4909, 0.005, CLMI_F64)
    rng = np.random.default_rng(3)
    for k in (FLD_S, PI_S):
        for f in range(2):
            lat.upload(k, f, 0, 0.3 * rng.standard_normal((N, N, N)))
    lat.set_background(aI=1.0, aSI=1.0, aIM=1.0, aDotI=0.7)
    lat.set_all_averages()
    lat.lf_init()
    lat.lf_evolve(20)
    lat.lf_sync()
    lat.vv_evolve(VV_WEIGHTS["VV2"], 10)
    h = hashlib.sha256()
    for k in (FLD_S, PI_S):
        for f in range(2):
            h.update(lat.download(k, f, 0).tobytes())
    h.update(repr(sorted(lat.background().items())).encode())
    return lat, h.hexdigest()


def test_second_process_evolves_alike(gpu):
    say("case resident in two processes")
    lat, want = evolve()  # this process holds the cooperative queue from here on
    code = (f"import sys; sys.path[:0] = [{str(ROOT)!r}, {str(ROOT / 'tests')!r}]\n"
            "from test_gpu_resident_processes import evolve\n"
            "lat, got = evolve()\nprint('hash', got)\nlat.close()\n")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert r.stdout.split()[-1] == want
    lat.close()
