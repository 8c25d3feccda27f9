"""Instances without a step in a batch's run: their states are left alone, also where the host finishes a step that
needed more iterations than were enqueued (iter_batch 1) while they are idle; the others run as on their own."""
import numpy as np
import pytest

from conftest import SMALL, dt_of
from dirac_hydrogen_code_amd import gade

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("first", [False, True])  # whether the idle ones have run before (a decided solve behind them)
@pytest.mark.parametrize("cfg", ["dipole", "nondipole_small"])
def test_idle_instances_keep_their_states(datadir, cfg, first, precision):
    print(f"[gpu] idle instances {cfg} first={first} precision={precision}", flush=True)
    d, dt, nl = datadir(cfg), dt_of(cfg), SMALL[cfg]["nl"]
    rng = np.random.default_rng(6)
    params = [(60.0, 50.0, 2.0, 0.0), (40.0, 50.0, 2.0, 1.0), (60.0, 50.0, 2.0, 2.0)]
    steps = [0, 4, 0]
    one, gp = gade.Propagator(d, nl, dt), gade.Propagator(d, nl, dt, batch=3)
    psi = rng.standard_normal((3, one.n)) + 1j * rng.standard_normal((3, one.n))
    for m in (one, gp):
        m.set_param("precision", precision)
    x = gade.DeviceArray.from_host(psi)
    if first:
        gp.cn_run_batch(x, params, 2, t0=0.03, tol=1e-12)
        psi = x.get().reshape(3, -1)
        gp.reset_workspace()
    gp.set_param("iter_batch", 1)
    it, _ = gp.cn_run_batch(x, params, 4, nsteps_b=steps, t0=0.05, tol=1e-12)
    assert it[1].max() >= 1
    y = gade.DeviceArray.from_host(psi[1])
    it1, _ = one.cn_run_batch(y, params[1:2], 4, t0=0.05, tol=1e-12)
    got = x.get().reshape(3, -1)
    assert np.array_equal(it[1], it1[0])
    for b, want in enumerate((psi[0], y.get(), psi[2])):
        assert np.array_equal(got[b].view(np.float64), want.view(np.float64)), b
