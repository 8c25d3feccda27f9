"""Eigen-projection of many blocks and of few rows: workgroups of fewer threads (no more than a block's eigenpairs need,
256 from 513 blocks on).  Against the projection formed here in 64 bit from the library's own eigenvectors; bar as
test_gpu_populations.py (1e-11 of a block's norm)."""
import os

import numpy as np
import pytest

import oracle as O
from dirac_hydrogen_code_amd import gade
from dirac_hydrogen_code_amd.couplings import generate
from test_gpu_populations import dense

pytestmark = pytest.mark.gpu


# 12 and 544 blocks of 16, 18, 62, 64 and 66 rows: one to three passes of 32 eigenpairs, with remainders
@pytest.mark.parametrize("nkappa,blocks", [(2, 12), (16, 544)])
@pytest.mark.parametrize("ns", [3, 4, 26, 27, 28])
def test_projection_of_many_blocks(tmp_path, nkappa, blocks, ns):
    print(f"[gpu] projection of {blocks} blocks of {2 * (ns + 5)}", flush=True)
    d = str(tmp_path)
    generate(d, nsplines=ns, nkappa=nkappa, nmu=0, nl=1, rbox=10.0, Z=1, intensity=10, omega=50.0, cycles=1)
    gp = gade.Propagator(d, 1, 2 * np.pi / 50 / 200)
    n = gp.blkdim
    assert (gp.nblk, n) == (blocks, 2 * (ns + 5))
    rng = np.random.default_rng(ns)
    psi = rng.standard_normal((blocks, n)) + 1j * rng.standard_normal((blocks, n))
    dpsi = gade.DeviceArray.from_host(psi)
    got = gp.populations(dpsi, per_block=True)
    amp = gp.psiev(dpsi).reshape(-1, n)
    gp.eig_write(d)
    ref, c2 = O.eigenpairs(d), 137.035999084 ** 2
    perm = O._read_csr(os.path.join(d, "H.csr"))[4]
    total = np.zeros(4)
    for k in {int(O.lib().or_ik(int(p))) for p in perm}:
        rows = [r for r in range(blocks) if O.lib().or_ik(int(perm[r])) == k]
        E = dense(os.path.join(d, f"evl{k}.mat"), False)[:, 0]
        V = dense(os.path.join(d, f"evc{k}.mat"), True)
        w = psi[rows] @ np.asarray(ref[k][2]).T
        c = w @ V.conj()
        p = np.abs(c) ** 2
        nrm = np.sum(psi[rows].conj() * w, axis=1).real
        want = np.stack([p[:, E < -c2].sum(1), p[:, (E >= -c2) & (E < 0)].sum(1), p[:, E >= 0].sum(1), nrm], 1)
        assert np.all(np.abs(got["per_block"][rows] - want) <= 1e-11 * nrm[:, None]), k
        assert np.all(np.abs(amp[rows] - c.conj()) <= 1e-11 * np.sqrt(nrm)[:, None]), k
        total += want.sum(0)
    for name, i in (("bound", 1), ("ionised", 2), ("norm", 3)):
        assert abs(got[name] - total[i]) <= 1e-11 * total[3]
