"""The training batch (loss and gradient of the learned guess's network) against the CPU oracle at the edges of its
kernels: one workgroup of 16 samples, up to 64 rows (four interleaved sums) and beyond, step counts that leave waves
of the gradient kernel without work or with a remainder, samples in any order, and the weights'
operand copies after a training step.  Bars: test_gpu_learned.py's (loss 1e-4, gradients 5e-3 per layer)."""
import numpy as np
import pytest

import lg_oracle as LG
from dirac_hydrogen_code_amd import gade
from test_gpu_learned import net_model, random_params, random_samples, say

pytestmark = pytest.mark.gpu


def check(gp, S, idx, mean, std):
    M = len(idx)
    ds = gade.DeviceArray.from_host(S.ravel())
    didx = gade.DeviceArray.from_host(idx.astype(np.int32))
    dg = gade.DeviceArray(LG.NPARAM, np.float32)
    loss = gp.lg_grad(ds, didx, M, dg)
    assert gp.lg_grad(ds, didx, M) == loss  # without a gradient buffer
    g = dg.get().astype(np.float64)
    p = gp.lg_get_params()
    T = S[idx]
    X = LG.standardize(T[:, :LG.IN].astype(np.float64), mean, std).astype(np.float32)
    Y, cache = LG.forward(p, X, quantized=True)
    lo, dY = LG.loss_and_dY(Y, T)
    go = LG.backward(p, cache, dY.astype(np.float32), quantized=True)
    assert abs(loss - lo) <= 1e-4 * abs(lo)
    for k, (fi, fo) in enumerate(LG.LAYERS):
        wo, bo = LG.OFFS[k]
        for a, b in ((g[wo:wo + fo * fi], go[wo:wo + fo * fi]), (g[bo:bo + fo], go[bo:bo + fo])):
            assert np.linalg.norm(a - b) <= 5e-3 * np.linalg.norm(b), k


@pytest.mark.parametrize("M", [16, 64, 80, 272, 1040])
def test_batch_edges(datadir, M):
    say(f"learned batch M={M}")
    rng = np.random.default_rng(M)
    gp = net_model(datadir)
    mean = rng.standard_normal(LG.IN).astype(np.float32)
    std = rng.uniform(0.5, 2.0, LG.IN).astype(np.float32)
    gp.lg_set_norm(mean, std)
    gp.lg_set_params(random_params(rng))
    S = random_samples(rng, min(M, 80) + 3, n=160)
    idx = rng.integers(0, len(S), M)
    check(gp, S, idx, mean, std)
    ds = gade.DeviceArray.from_host(S.ravel())
    gp.lg_train(ds, gade.DeviceArray.from_host(idx.astype(np.int32)), M, 1, 1e-3)
    check(gp, S, idx, mean, std)
