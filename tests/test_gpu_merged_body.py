"""The device-driven BiCGSTAB body against the kernels it merges.

The host loop runs one kernel per operation: p, solve, product, alpha, s, solve, product, w, x and r.  The device
loop runs eight launches a body: the vector steps and alpha inside the preconditioner solves (one, two or four blocks
of one kappa per workgroup), the dot products on the products' sums, w inside the update.  Sums keep their order, so
the two agree bit for bit; a batch, whose workgroups mix instances that have finished with ones that go on, agrees
with its instances run alone."""
import numpy as np
import pytest

from conftest import SMALL, dt_of
from dirac_hydrogen_code_amd import gade
from dirac_hydrogen_code_amd.couplings import generate

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def couplings(tmp_path_factory):
    """Blocks of one instance: below 320, to 1280 and from 1280 a workgroup of the solve takes one, two, four."""
    def get(nkappa, nsplines, nl):
        if (nkappa, nsplines, nl) not in made:
            d = str(tmp_path_factory.mktemp("body"))
            generate(d, nsplines=nsplines, nkappa=nkappa, nmu=0, nl=nl, rbox=10.0, Z=1, intensity=10, omega=50.0, cycles=1)
            made[nkappa, nsplines, nl] = d
        return made[nkappa, nsplines, nl]
    made = {}
    return get


# 40, 112, 364 and 1300 blocks; radial sizes of one to four levels of 16 rows, with remainders
@pytest.mark.parametrize("nkappa,nsplines,nl,blocks", [(4, 3, 1, 40), (7, 27, 3, 112), (13, 12, 1, 364),
                                                       (13, 19, 2, 364), (25, 8, 1, 1300)])
def test_device_body_equals_separate_kernels(couplings, nkappa, nsplines, nl, blocks):
    print(f"[gpu] merged body {blocks} blocks of {2 * (nsplines + 5)}, {nl} multipoles", flush=True)
    d, dt = couplings(nkappa, nsplines, nl), 2 * np.pi / 50 / 40
    gp = gade.Propagator(d, nl, dt)
    assert gp.nblk == blocks
    rng = np.random.default_rng(blocks)
    psi = rng.standard_normal(gp.n) + 1j * rng.standard_normal(gp.n)
    out, launches = {}, {}
    for dev in (0, 1):
        gp.set_param("device_loop", dev)
        gp.reset_workspace()
        x = gade.DeviceArray.from_host(psi)
        gp.profile(["blas1"])
        before = gp.profile_get("blas1")[1]
        it, tols, _ = gp.cn_run(x, 60.0, 50.0, 1.0, 6, t0=0.03, tol=1e-12, timing=False)
        launches[dev] = gp.profile_get("blas1")[1] - before
        gp.profile(False)
        out[dev] = x.get(), it, tols
    assert out[0][1].min() >= 1  # at least two bodies a step
    # the vector operations of the host loop are launches of their own: one at the start of a solve, five a body
    assert launches[0] == np.sum(1 + 5 * (out[0][1] + 1))
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(np.asarray(a).view(np.uint8), np.asarray(b).view(np.uint8))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("cfg,batch", [("dipole", 9), ("dipole", 33)])  # 360 and 1320 blocks
def test_mixed_workgroups_equal_single_runs(datadir, cfg, batch, precision):
    print(f"[gpu] merged body batch of {batch} precision={precision}", flush=True)
    d, dt, nl = datadir(cfg), dt_of(cfg), SMALL[cfg]["nl"]
    one, gp = gade.Propagator(d, nl, dt), gade.Propagator(d, nl, dt, batch=batch)
    rng = np.random.default_rng(batch)
    psi = rng.standard_normal((batch, one.n)) + 1j * rng.standard_normal((batch, one.n))
    params = [(float(rng.uniform(1, 80)), 50.0, 1.0, float(rng.uniform(0, 6))) for _ in range(batch)]
    steps = [int(rng.integers(0, 6)) for _ in range(batch)]
    steps[0] = 5
    for m in (one, gp):
        m.set_param("precision", precision)
    x = gade.DeviceArray.from_host(psi)
    it, tols = gp.cn_run_batch(x, params, 5, nsteps_b=steps, t0=0.03, tol=1e-12)
    got = x.get().reshape(batch, -1)
    counts = set()
    for b in range(batch):
        y = gade.DeviceArray.from_host(psi[b])
        one.reset_workspace()
        if steps[b]:
            it1, tol1 = one.cn_run_batch(y, params[b:b + 1], steps[b], t0=0.03, tol=1e-12)
            assert np.array_equal(it[b, :steps[b]], it1[0]) and np.array_equal(tols[b, :steps[b]], tol1[0]), b
            counts.update(it1[0])
        assert np.array_equal(got[b].view(np.float64), y.get().view(np.float64)), b
    assert len(counts) > 1  # some instances have finished a solve while others go on
