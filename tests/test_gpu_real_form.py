"""The banded products' real and complex forms against the oracle.

The couplings of the physics are real up to one common factor of the angular ones (i, or 1 for files that carry it
elsewhere) and f(t) is real: the kernels then run on real coefficients.  Anything else (complex radial couplings,
angular couplings of no common phase, complex f(t)) runs the complex form.  Both must give the oracle's products.
Bar: max-norm relative 1e-13, as for every operator product (tests/test_gpu_parity.py).
"""
import os
import shutil

import numpy as np
import pytest

import oracle as O
from dirac_hydrogen_code_amd import gade
from dirac_hydrogen_code_amd.couplings import csr_read, csr_write, generate

pytestmark = pytest.mark.gpu

NL = 2
# radial halves of 15, 64, 65 and 133 functions: below, at and past one 64-output segment, and a ragged third
SPLINES = (10, 59, 60, 128)
SHAPES = ((4, 1, 2, 1), (8, 2, 1, 0), (4, 4, 2, 0), (16, 1, 2, 1))  # rows, outputs, halves, fused


@pytest.fixture(scope="module")
def variants(tmp_path_factory):
    """Couplings of each size as generated ("i"), with the angular ones turned real ("1") or to no common phase
    ("mixed": the two angular kinds a quarter turn and a third apart), and with complex radial couplings ("g")."""
    base = str(tmp_path_factory.mktemp("forms"))
    rng = np.random.default_rng(5)

    def scale(d, prefix, factor):
        for f in sorted(os.listdir(d)):
            if f.startswith(prefix) and f.endswith(".csr"):
                m = csr_read(os.path.join(d, f))
                csr_write(os.path.join(d, f), m["Ap"], m["Ai"], m["Ax"] * factor(len(m["Ax"])))

    def get(ns, kind):
        d = os.path.join(base, f"{ns}_{kind}")
        if not os.path.isdir(d):
            if kind == "i":
                generate(d, nsplines=ns, nkappa=3, nmu=0, nl=NL, rbox=12.0, Z=1, intensity=10, omega=50.0, cycles=1)
                return d
            shutil.copytree(get(ns, "i"), d)
            if kind == "1":
                scale(d, "H0l", lambda n: -1j)
                scale(d, "H1l", lambda n: -1j)
            elif kind == "mixed":
                scale(d, "H1l", lambda n: np.exp(2j * np.pi / 3))
            else:
                scale(d, "g", lambda n: 1 + 0.3j * rng.standard_normal(n))
        return d

    return get


@pytest.mark.parametrize("kind", ["i", "1", "mixed", "g"])
@pytest.mark.parametrize("ns", SPLINES)
def test_products_of_real_and_complex_couplings(variants, ns, kind):
    print(f"[gpu] real form ns={ns} couplings={kind}", flush=True)
    d, dt = variants(ns, kind), 2 * np.pi / 50 / 200
    om, gp = O.Model(d, NL, dt, nthreads=4), gade.Propagator(d, NL, dt)
    rng = np.random.default_rng(ns)
    x = rng.standard_normal(gp.n) + 1j * rng.standard_normal(gp.n)
    y0 = rng.standard_normal(gp.n) + 1j * rng.standard_normal(gp.n)
    dx, dy = gade.DeviceArray.from_host(x), gade.DeviceArray(gp.n)
    shapes = (None,) + SHAPES  # the model's own shape first
    for shape in shapes:
        if shape:
            gp.set_param("ang_fused", 0)
            gp.set_param("dia_outputs", 1)
            for name, value in zip(("dia_rows", "dia_outputs", "dia_halves", "ang_fused"), shape):
                gp.set_param(name, value)
        # real f(t), complex f(t), and back: each product runs in the form of the f(t) set last
        for f in (gade.pulse(10, 50, 1, 0.02), rng.standard_normal(6) + 1j * rng.standard_normal(6),
                  rng.standard_normal(6) + 0j):
            om.timedep(f)
            gp.set_time(f)
            S, H = om.apply(x, "S"), om.apply(x, "H")
            for cH, beta, want in ((1.0, 0.0, S + H), (-1.0, 0.5, S - H + 0.5 * y0), (0.0, 0.0, S)):
                dy.upload(y0)
                gp.apply(dx, dy, cH=cH, beta=beta)
                err = np.abs(dy.get() - want).max() / np.abs(want).max()
                assert err <= 1e-13, (shape, cH, err)
