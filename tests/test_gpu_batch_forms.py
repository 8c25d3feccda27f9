"""A batch whose instances stop at different steps: the G-sums of each instance stay those of the f(t) it had last,
whatever form (real or complex) the other instances' steps and later parameter changes bring.

Bars: operator products against the oracle at each instance's own f(t), max-norm relative 1e-13
(as tests/test_gpu_parity.py); the forms give the same trajectories bit for bit."""
import numpy as np
import pytest

import oracle as O
from conftest import dt_of
from dirac_hydrogen_code_amd import gade

pytestmark = pytest.mark.gpu

LMAX = {"dipole": 1, "nondipole_small": 4}
PARAMS = [(10.0, 50.0, 2.0, 0.3), (25.0, 45.0, 2.0, 1.0), (5.0, 55.0, 2.0, 0.0)]
T0 = 0.05


def batch_of(datadir, cfg, held, nsteps_b, precision=0):
    """A batch with f(t) = held, run for nsteps_b steps: the model, its states and the f(t) of each instance."""
    d, dt = datadir(cfg), dt_of(cfg)
    gp = gade.Propagator(d, LMAX[cfg], dt, batch=len(PARAMS))
    gp.set_param("precision", precision)
    gp.set_time_batch(np.array(held))
    psi0, _ = gade.read_psi0(d, gp.n)
    x = gade.DeviceArray.from_host(np.tile(psi0, len(PARAMS)))
    gp.cn_run_batch(x, PARAMS, max(nsteps_b), nsteps_b=nsteps_b, t0=T0, tol=1e-12)
    f = [gade.pulse_cep(*PARAMS[b], T0 + nsteps_b[b] * dt) if nsteps_b[b] else held[b] for b in range(len(PARAMS))]
    return gp, x.get(), f


def check(gp, om, f, what):
    n = gp.n * len(f)
    rng = np.random.default_rng(2)
    x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    dx, dy = gade.DeviceArray.from_host(x), gade.DeviceArray(n)
    gp.apply(dx, dy)
    for b, (xb, yb) in enumerate(zip(x.reshape(len(f), -1), dy.get().reshape(len(f), -1))):
        om.timedep(f[b])
        want = om.apply(xb, "S") + om.apply(xb, "H")
        err = np.abs(yb - want).max() / np.abs(want).max()
        assert err <= 1e-13, (what, b, err)


# which instances hold a complex f(t) before the run, and the steps of each
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("cfg,cplx,nsteps_b", [
    ("dipole", (1, 1, 1), [0, 5, 3]),           # a complex one is kept: the run has to leave it complex
    ("nondipole_small", (0, 1, 0), [4, 0, 4]),
    ("dipole", (1, 0, 1), [4, 0, 4]),           # a real one is kept while the others' complex sums go
    ("nondipole_small", (1, 0, 0), [3, 0, 12]),
    ("nondipole_small", (0, 0, 0), [0, 2, 9]),  # no change of form
])
def test_instances_without_a_step_keep_their_sums(datadir, cfg, cplx, nsteps_b, precision):
    print(f"[gpu] batch forms {cfg} {cplx} {nsteps_b} precision={precision}", flush=True)
    rng = np.random.default_rng(sum(nsteps_b))
    held = [rng.standard_normal(6) + 1j * c * rng.standard_normal(6) for c in cplx]
    om = O.Model(datadir(cfg), LMAX[cfg], dt_of(cfg), nthreads=4)
    gp, psi, f = batch_of(datadir, cfg, held, nsteps_b, precision)
    check(gp, om, f, "after the run")
    _, want, _ = batch_of(datadir, cfg, [h.real + 0j for h in held], nsteps_b, precision)
    assert np.array_equal(psi.view(np.float64), want.view(np.float64))


@pytest.mark.parametrize("name,values", [("ang_list", (0, 1)), ("radial_mfma", (1, 0))])
@pytest.mark.parametrize("cfg", ["dipole", "nondipole_small"])
def test_kernel_switch_keeps_every_instance(datadir, cfg, name, values):
    """ang_list and radial_mfma change the layout of the G-sums, not the f(t) that each instance stopped at."""
    print(f"[gpu] {name} after a batch of unequal lengths {cfg}", flush=True)
    held = [gade.pulse(10, 50, 2, 0.01)] * len(PARAMS)
    om = O.Model(datadir(cfg), LMAX[cfg], dt_of(cfg), nthreads=4)
    gp, _, f = batch_of(datadir, cfg, held, [9, 0, 4])
    for value in values:
        gp.set_param(name, value)
        check(gp, om, f, f"{name} {value}")
