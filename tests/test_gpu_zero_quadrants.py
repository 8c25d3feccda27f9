"""Real radial couplings with and without the zero quadrants of a dual-kinetic-balance basis.

The generated couplings have them (the kernels then leave the vanishing products out: covered by
test_gpu_real_form.py, every product against the oracle); a single entry outside them must bring the full real form
back, whichever coupling and quadrant it is in.  Bar: max-norm relative 1e-13 (tests/test_gpu_parity.py)."""
import os

import numpy as np
import pytest

import oracle as O
from dirac_hydrogen_code_amd import gade
from dirac_hydrogen_code_amd.couplings import csr_read, csr_write, generate
from test_gpu_real_form import SHAPES

pytestmark = pytest.mark.gpu
NL = 2


# ns: radial halves of 15, 64 and 65 functions; the coupling n and quadrant (h, h') filled, or every one
@pytest.mark.parametrize("ns,n,h,hp", [(10, 1, 0, 0), (59, 1, 0, 1), (60, 2, 0, 1), (10, 2, 1, 1), (60, 3, 0, 0),
                                       (10, 3, 0, 1), (59, 3, 1, 1), (60, 0, -1, -1)])
def test_filled_quadrants(tmp_path, ns, n, h, hp):
    print(f"[gpu] zero quadrants ns={ns} n={n} quadrant=({h},{hp})", flush=True)
    d, dt = str(tmp_path), 2 * np.pi / 50 / 200
    generate(d, nsplines=ns, nkappa=3, nmu=0, nl=NL, rbox=12.0, Z=1, intensity=10, omega=50.0, cycles=1)
    rng = np.random.default_rng(ns)
    for f in sorted(os.listdir(d)):
        if not (f.startswith("g") and f.endswith(".csr")):
            continue
        m = csr_read(os.path.join(d, f))
        nh = m["n"] // 2
        row = np.repeat(np.arange(m["n"]), np.diff(m["Ap"]))
        zero = m["Ax"] == 0
        if h >= 0:  # one entry of one coupling
            pick = np.flatnonzero(zero & (row // nh == h) & (m["Ai"] // nh == hp))
            zero = np.zeros_like(zero)
            if f == f"g{n}a2l1.csr":
                zero[pick[len(pick) // 2]] = True
        scale = np.abs(m["Ax"]).max()
        csr_write(os.path.join(d, f), m["Ap"], m["Ai"], m["Ax"] + zero * scale * rng.standard_normal(len(row)))
    om, gp = O.Model(d, NL, dt, nthreads=4), gade.Propagator(d, NL, dt)
    x = rng.standard_normal(gp.n) + 1j * rng.standard_normal(gp.n)
    dx, dy = gade.DeviceArray.from_host(x), gade.DeviceArray(gp.n)
    for shape in (None,) + SHAPES:
        if shape:
            gp.set_param("ang_fused", 0)
            gp.set_param("dia_outputs", 1)
            for name, value in zip(("dia_rows", "dia_outputs", "dia_halves", "ang_fused"), shape):
                gp.set_param(name, value)
        for f in (gade.pulse(10, 50, 1, 0.02), rng.standard_normal(6) + 1j * rng.standard_normal(6),
                  rng.standard_normal(6) + 0j):
            om.timedep(f)
            gp.set_time(f)
            ref = om.apply(x, "S") + om.apply(x, "H")
            gp.apply(dx, dy)
            assert np.abs(dy.get() - ref).max() <= 1e-13 * np.abs(ref).max(), (shape, f)
