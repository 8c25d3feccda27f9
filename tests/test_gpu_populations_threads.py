"""Populations of several states from several threads on one model: each call returns its own state's sums, bit for
bit those of the same call alone (the kernel's sums have a fixed order)."""
import threading

import numpy as np
import pytest

from conftest import dt_of
from dirac_hydrogen_code_amd import gade

pytestmark = pytest.mark.gpu


def test_populations_from_threads(datadir):
    d, dt = datadir("dipole"), dt_of("dipole")
    gp = gade.Propagator(d, 1, dt)
    print("[gpu] populations from four threads", flush=True)
    rng = np.random.default_rng(4)
    x = [gade.DeviceArray.from_host(rng.standard_normal(gp.n) + 1j * rng.standard_normal(gp.n)) for _ in range(4)]
    alone = [gp.populations(v, per_block=True)["per_block"].copy() for v in x]
    wrong = []

    def call(k):
        for _ in range(200):
            got = gp.populations(x[k], per_block=True)["per_block"]
            if not np.array_equal(got, alone[k]):
                wrong.append(k)

    threads = [threading.Thread(target=call, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, len(wrong)
