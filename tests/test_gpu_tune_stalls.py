"""A tuned model goes on as it would have without tuning: the candidates that enqueue too few iterations a step leave
no spare ones behind, neither for the candidates after them nor for the next run."""
import pytest

from conftest import SMALL, dt_of
from dirac_hydrogen_code_amd import gade

pytestmark = pytest.mark.gpu

DEFAULTS = dict(window=8, iter_batch=0, graph=1)


@pytest.mark.parametrize("cfg", ["dipole", "nondipole_small"])
def test_no_spare_iterations_after_tuning(datadir, cfg):
    print(f"[gpu] iterations enqueued after tuning {cfg}", flush=True)
    d, dt = datadir(cfg), dt_of(cfg)
    solves = {}
    for tune in (0, 1):
        gp = gade.Propagator(d, SMALL[cfg]["nl"], dt)
        assert {k: gp.get_param(k) for k in DEFAULTS} == DEFAULTS
        psi0, _ = gade.read_psi0(d, gp.n)
        x = gade.DeviceArray.from_host(psi0)
        if tune:
            _, rows = gp.autotune(x, [(10.0, 50.0, 2.0, 0.0)], 3, t0=0.05, reps=1)
            assert any(r["iter_batch"] == 1 for r in rows)
            for k, v in DEFAULTS.items():
                gp.set_param(k, v)
        gp.profile(["psolve"])
        it, _, _ = gp.cn_run(x, 10.0, 50.0, 2.0, 24, t0=0.05, tol=1e-12, timing=False)
        solves[tune] = gp.profile_get("psolve")[1]
        assert it.max() == 1  # two bodies a step: one enqueued is too few, the usual two are enough
    assert solves[0] == solves[1]
