"""Device memory of a training batch: what its two launches use, not the forward pass's FP32 buffers."""
import ctypes as C

import numpy as np
import pytest

import lg_oracle as LG
from dirac_hydrogen_code_amd import gade
from test_gpu_learned import net_model, random_params, random_samples, say

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert gade.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0  # from the runtime that the library is linked to
    return free.value


def test_training_buffers(datadir):
    M = 16384
    say(f"memory of a training batch of {M}")
    rng = np.random.default_rng(1)
    gp = net_model(datadir)
    gp.lg_set_params(random_params(rng))
    S = np.resize(random_samples(rng, 64), (M, LG.SAMPLE)).astype(np.float32)
    ds, didx = gade.DeviceArray.from_host(S.ravel()), gade.DeviceArray.from_host(rng.permutation(M).astype(np.int32))
    gp.lg_grad(ds, didx, 16)
    before = free_bytes()
    loss = gp.lg_grad(ds, didx, M)
    used = before - free_bytes()
    # bf16 inputs, three activations and four gradients, FP32 bias sums of every fourth row, losses; ten allocations
    # of up to 2 MiB more each
    need = M * (2 * LG.IN + 2 * 256 * 7 + 4 * (3 * 256 + LG.OUT) // 4 + 4)
    assert used <= need + 10 * 2 ** 21, (used, need)
    assert np.isfinite(loss)
    x = gade.DeviceArray.from_host(np.ascontiguousarray(S[:, :LG.IN]).ravel())
    y = gade.DeviceArray(M * LG.OUT, np.float32)
    gp.lg_forward(x, M, y)  # which allocates them
    assert np.all(np.isfinite(y.get()))
    assert gp.lg_grad(ds, didx, M) == loss
