"""The assembled matrix on both sides of 11 multipoles, from which its kernel has sixteen waves instead of four: block
rows with fewer Hall entries than waves and with more.  Bar: max-norm relative 1e-13 (test_gpu_assembled.py)."""
import numpy as np
import pytest

import oracle as O
from dirac_hydrogen_code_amd import gade
from dirac_hydrogen_code_amd.couplings import generate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nl", [10, 11])
@pytest.mark.parametrize("nkappa", [1, 2, 3])
def test_assembled_waves(tmp_path, nkappa, nl):
    print(f"[gpu] assembled nkappa={nkappa} nl={nl}", flush=True)
    d, dt = str(tmp_path), 2 * np.pi / 50 / 200
    generate(d, nsplines=8, nkappa=nkappa, nmu=0, nl=nl, rbox=10.0, Z=1, intensity=10, omega=50.0, cycles=1)
    om, gp = O.Model(d, nl, dt, nthreads=4), gade.Propagator(d, nl, dt)
    rng = np.random.default_rng(nl)
    f = rng.standard_normal(6) + 1j * rng.standard_normal(6)
    om.timedep(f)
    gp.set_time(f)
    gp.assembled_timedep()
    want = om.hfull_values()
    got = gp.assembled_get(submap=False)[3]
    assert np.abs(got - want).max() <= 1e-13 * np.abs(want).max()
