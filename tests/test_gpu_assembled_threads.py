"""The assembled matrix from several threads on one new model, each into its own buffer: nothing is set up by the
first call that the others could find half done.  The values are those of a single call, bit for bit."""
import ctypes as C
import threading

import numpy as np
import pytest

from conftest import dt_of
from dirac_hydrogen_code_amd import gade

pytestmark = pytest.mark.gpu


def test_assemble_into_from_threads(datadir):
    d, dt = datadir("nondipole_small"), dt_of("nondipole_small")
    f = gade.pulse(10, 50, 2, 0.07)
    one = gade.Propagator(d, 4, dt)
    one.set_time(f)
    one.assembled_timedep()
    Ap, _, _, want = one.assembled_get(submap=False)
    dAp = gade.DeviceArray.from_host(Ap)
    for trial in range(3):
        print(f"[gpu] assemble from four threads, model {trial}", flush=True)
        gp = gade.Propagator(d, 4, dt)
        gp.set_time(f)
        out = [gade.DeviceArray(len(want)) for _ in range(4)]
        rc = [None] * 4

        def call(k):
            rc[k] = gade.lib().gade_assembled_timedep_into(C.c_void_p(gp.ptr), C.c_void_p(dAp.ptr),
                                                           C.c_void_p(out[k].ptr))

        threads = [threading.Thread(target=call, args=(k,)) for k in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert rc == [0] * 4
        for o in out:
            assert np.array_equal(o.get().view(np.float64), want.view(np.float64))
