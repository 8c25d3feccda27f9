"""The network's forward pass of rows against the CPU oracle around the sizes where its kernels change: four waves per
tile up to 64 rows, one with six steps in flight below 1024, one with two from there.  Bar: test_gpu_learned.py's 3e-4,
in the norm (an activation that the two sides round to different bf16 neighbours moves one entry, and more rows have
more of those)."""
import numpy as np
import pytest

import lg_oracle as LG
from dirac_hydrogen_code_amd import gade
from test_gpu_learned import net_model, random_params, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [16, 64, 80, 1008, 1024, 1040])
def test_forward_rows(datadir, M):
    say(f"forward of {M} rows")
    rng = np.random.default_rng(M)
    gp = net_model(datadir)
    p = random_params(rng)
    mean, std = rng.standard_normal(LG.IN).astype(np.float32), (0.5 + rng.random(LG.IN)).astype(np.float32)
    gp.lg_set_norm(mean, std)
    gp.lg_set_params(p)
    x = (mean + std * rng.standard_normal((M, LG.IN))).astype(np.float32)
    dx, dy = gade.DeviceArray.from_host(x.ravel()), gade.DeviceArray(M * LG.OUT, np.float32)
    gp.lg_forward(dx, M, dy)
    want, _ = LG.forward(p, LG.standardize(x.astype(np.float64), mean, std).astype(np.float32), quantized=True)
    got = dy.get().reshape(M, LG.OUT)
    assert np.linalg.norm(got - want) <= 3e-4 * np.linalg.norm(want)
