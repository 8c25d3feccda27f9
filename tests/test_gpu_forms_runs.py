"""CN runs and products of the banded kernels' forms: real couplings with and without the zero quadrants, angular
couplings real, imaginary or of no common phase, complex radial couplings, and the Hall rows' parameter.

Every form takes the same kernel shapes (rows, outputs, halves, angular phase inside or not) with the same sums: the
shapes agree bit for bit, in the paired product and the FP32 inner solves of a run too.  Against the oracle: products
max-norm relative 1e-13, trajectories 1e-9 (as tests/test_gpu_parity.py)."""
import os
import shutil

import numpy as np
import pytest

import oracle as O
from dirac_hydrogen_code_amd import gade
from dirac_hydrogen_code_amd.couplings import csr_read, csr_write
from test_gpu_real_form import NL, variants  # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu

DT = 2 * np.pi / 50 / 200
SHAPES = ((4, 1, 2, 1), (4, 1, 1, 1), (4, 1, 1, 0), (4, 1, 2, 0), (8, 1, 1, 1), (8, 1, 2, 0), (8, 2, 2, 1),
          (8, 2, 1, 0), (4, 2, 1, 1), (4, 2, 2, 0), (16, 1, 2, 1), (16, 1, 1, 0), (4, 4, 1, 0), (4, 4, 2, 0))


def set_shape(gp, shape):
    gp.set_param("ang_fused", 0)
    gp.set_param("dia_outputs", 1)
    for name, value in zip(("dia_rows", "dia_outputs", "dia_halves", "ang_fused"), shape):
        gp.set_param(name, value)


@pytest.fixture(scope="module")
def couplings(variants):
    """The couplings of test_gpu_real_form.py, and "full": real ones with an entry outside the zero quadrants."""
    def get(ns, kind):
        if kind != "full":
            return variants(ns, kind)
        d = variants(ns, "i") + "_full"
        if not os.path.isdir(d):
            shutil.copytree(variants(ns, "i"), d)
            f = os.path.join(d, "g1a2l1.csr")
            m = csr_read(f)
            half = m["n"] // 2
            row = np.repeat(np.arange(m["n"]), np.diff(m["Ap"]))
            outside = np.flatnonzero((m["Ax"] == 0) & (row < half) & (m["Ai"] < half))
            m["Ax"] = m["Ax"].copy()
            m["Ax"][outside[len(outside) // 2]] = 0.1 * np.abs(m["Ax"]).max()
            csr_write(f, m["Ap"], m["Ai"], m["Ax"])
        return d
    return get


@pytest.mark.parametrize("batch,precision", [(1, 0), (1, 1), (3, 0), (3, 1)])
@pytest.mark.parametrize("kind", ["i", "full", "1", "mixed", "g"])
def test_runs_match_oracle_and_each_other(couplings, kind, batch, precision):
    print(f"[gpu] forms: runs, couplings={kind} batch={batch} precision={precision}", flush=True)
    d, steps = couplings(10, kind), 6
    gp = gade.Propagator(d, NL, DT, batch=batch)
    gp.set_param("precision", precision)
    psi0, _ = gade.read_psi0(d, gp.n)
    pulses = [(10.0 + 5 * b, 50.0, 1.0 + b, 0.0) for b in range(batch)]
    first = None
    for shape in (None,) + SHAPES:
        if shape:
            set_shape(gp, shape)
        x = gade.DeviceArray.from_host(np.tile(psi0, batch))
        gp.reset_workspace()
        it, tols = gp.cn_run_batch(x, pulses, steps, tol=1e-12)
        got = x.get().reshape(batch, -1)
        assert np.all(tols <= 1e-12)
        if first is None:
            first = got, it, tols
            for b, (e0, w, c, _) in enumerate(pulses):
                want = O.Model(d, NL, DT, nthreads=4).cn_run(psi0, e0, w, c, steps, tol=1e-12)[0]
                assert np.linalg.norm(got[b] - want) <= 1e-9 * np.linalg.norm(want), b
        for a, b in zip((got, it, tols), first):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), shape


# radial halves of 15, 64 and 133 functions
@pytest.mark.parametrize("ns", [10, 59, 128])
@pytest.mark.parametrize("kind,cplx,ang_list", [("i", True, 1), ("mixed", False, 1), ("g", False, 1), ("i", False, 0),
                                                ("full", False, 1)])
def test_every_form_has_every_shape(couplings, ns, kind, cplx, ang_list):
    """The shape that is set is the one that runs: with the angular phase inside there is no angular kernel."""
    print(f"[gpu] forms: shapes ns={ns} couplings={kind} complex f={cplx} ang_list={ang_list}", flush=True)
    d = couplings(ns, kind)
    om, gp = O.Model(d, NL, DT, nthreads=4), gade.Propagator(d, NL, DT)
    gp.set_param("ang_list", ang_list)
    rng = np.random.default_rng(ns)
    f = gade.pulse(10, 50, 1, 0.02) * (1 + 0.3j if cplx else 1)
    x = rng.standard_normal(gp.n) + 1j * rng.standard_normal(gp.n)
    dx, dy = gade.DeviceArray.from_host(x), gade.DeviceArray(gp.n)
    om.timedep(f)
    gp.set_time(f)
    want, first = om.apply(x, "S") + om.apply(x, "H"), None
    for shape in (None,) + SHAPES:
        if shape:
            set_shape(gp, shape)
        gp.profile(["angular"])
        before = gp.profile_get("angular")[1]
        gp.apply(dx, dy)
        launches = gp.profile_get("angular")[1] - before
        gp.profile(False)
        assert launches == (0 if shape is None or shape[3] else 1), shape
        got = dy.get()
        if first is None:
            first = got
            assert np.abs(got - want).max() <= 1e-13 * np.abs(want).max()
        assert np.array_equal(got.view(np.float64), first.view(np.float64)), shape
