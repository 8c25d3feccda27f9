"""The banded kernels' shape parameters: what get_param returns is what runs, a setter changes its own parameter, and
the autotuner leaves alone what it does not tune."""
import numpy as np
import pytest

from conftest import SMALL, dt_of
from dirac_hydrogen_code_amd import gade

pytestmark = pytest.mark.gpu

NAMES = ("dia_rows", "dia_outputs", "dia_halves", "ang_fused")


def model(datadir, cfg="nondipole_small"):
    return gade.Propagator(datadir(cfg), SMALL[cfg]["nl"], dt_of(cfg))


def shape(gp):
    return tuple(gp.get_param(n) for n in NAMES)


def angular_launches(gp):
    """Angular kernels in one product: none with the phase inside the radial kernel."""
    dx, dy = gade.DeviceArray(gp.n), gade.DeviceArray(gp.n)
    dx.zero()
    gp.profile(["angular"])
    gp.apply(dx, dy)
    n = gp.profile_get("angular")[1]
    gp.profile(False)
    return n


def test_reported_shape_is_the_one_that_runs(datadir):
    print("[gpu] shape parameters", flush=True)
    gp = model(datadir)
    gp.set_time(gade.pulse(10, 50, 2, 0.05))
    assert shape(gp) == (4, 1, 2, 1) and angular_launches(gp) == 0
    for name, value in zip(NAMES, shape(gp)):  # the reported values change nothing
        gp.set_param(name, value)
        assert shape(gp) == (4, 1, 2, 1) and angular_launches(gp) == 0
    gp.set_param("dia_halves", 1)
    assert shape(gp) == (4, 1, 1, 1) and angular_launches(gp) == 0
    gp.set_param("dia_outputs", 2)
    assert shape(gp) == (4, 2, 1, 1) and angular_launches(gp) == 0
    gp.set_param("ang_fused", 0)
    assert shape(gp) == (4, 2, 1, 0) and angular_launches(gp) == 1
    gp.set_param("dia_outputs", 1)
    gp.set_param("dia_rows", 8)
    assert shape(gp) == (8, 1, 1, 0) and angular_launches(gp) == 1


def test_shape_without_a_fused_form(datadir):
    """(4,4) has none: a default follows the shape and comes back with it, a set one and the shape refuse each other."""
    print("[gpu] shape parameters: (4,4)", flush=True)
    gp = model(datadir)
    gp.set_param("dia_outputs", 4)
    assert shape(gp) == (4, 4, 2, 0) and angular_launches(gp) == 1
    with pytest.raises(gade.GadeError):
        gp.set_param("ang_fused", 1)
    gp.set_param("dia_outputs", 1)
    assert shape(gp) == (4, 1, 2, 1) and angular_launches(gp) == 0
    gp.set_param("ang_fused", 1)
    with pytest.raises(gade.GadeError):
        gp.set_param("dia_outputs", 4)
    assert shape(gp) == (4, 1, 2, 1)
    with pytest.raises(gade.GadeError):
        gp.set_param("dia_outputs", 3)


def test_tuning_the_matrix_core_form_keeps_the_shape(datadir):
    print("[gpu] shape parameters: tuning with radial_mfma", flush=True)
    gp = model(datadir)
    psi0, _ = gade.read_psi0(gp.directory, gp.n)
    x = gade.DeviceArray.from_host(psi0)
    gp.set_param("radial_mfma", 1)
    _, rows = gp.autotune(x, [(10.0, 50.0, 2.0, 0.0)], 3, t0=0.05, reps=1)
    assert {tuple(r[n] for n in NAMES) for r in rows} == {(4, 1, 2, 1)}
    assert shape(gp) == (4, 1, 2, 1)
    gp.set_param("radial_mfma", 0)
    assert angular_launches(gp) == 0
    gp.set_param("dia_outputs", 4)  # the form was not tuned: it follows the shape still
    assert shape(gp) == (4, 4, 2, 0)


@pytest.mark.parametrize("cfg", ["dipole", "nondipole_small"])
def test_tuned_shape_is_kept(datadir, cfg):
    print(f"[gpu] shape parameters: tuned {cfg}", flush=True)
    gp = model(datadir, cfg)
    psi0, _ = gade.read_psi0(gp.directory, gp.n)
    x = gade.DeviceArray.from_host(psi0)
    chosen, rows = gp.autotune(x, [(10.0, 50.0, 2.0, 0.0)], 3, t0=0.05, reps=1)
    best = tuple(rows[chosen][n] for n in NAMES)
    assert shape(gp) == best
    assert len({tuple(r[n] for n in NAMES) + (r["ang_lb"],) for r in rows[:46]}) == 46
    gp.set_param("dia_halves", best[2])
    assert shape(gp) == best
    assert np.isfinite(gp.snorm(x))
