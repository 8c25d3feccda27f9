"""The block preconditioner with several blocks of one factor per workgroup, through its C entry points."""
import ctypes as C

import numpy as np
import pytest

from dirac_hydrogen_code_amd import gade
from test_gpu_blocklu import banded_blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nblk,n,band", [(320, 17, 6), (321, 17, 6), (325, 33, 7), (1279, 16, 5), (1281, 40, 9),
                                         (1400, 1100, 4)])
def test_blocks_sharing_a_workgroup(nblk, n, band):
    """Many blocks: two or four of one factor per workgroup (the counts around the change, group sizes that leave
    padding, and blocks too tall for four of them in LDS).  Every block equals its dense solve to 1e-12."""
    rng = np.random.default_rng(nblk + n)
    blocks, mask = banded_blocks(n, band, 3, rng)
    which = rng.integers(0, 3, nblk)
    a, c = np.nonzero(mask)
    Ap = np.concatenate([[0], np.cumsum(np.tile(mask.sum(1), nblk))]).astype(np.int32)
    Ai = (np.arange(nblk)[:, None] * n + c[None, :]).astype(np.int32).ravel()
    Axr = np.ascontiguousarray(np.stack([blocks[q][a, c] for q in which]).ravel()).view(np.float64)
    L = gade.lib()
    L.gade_blocklu_create.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.POINTER(C.c_void_p)]
    L.gade_blocklu_solve.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p]
    L.gade_blocklu_destroy.argtypes = [C.c_void_p]
    lu = C.c_void_p()
    gade.check(L.gade_blocklu_create(nblk, n, Ap.ctypes.data, Ai.ctypes.data, Axr.ctypes.data, C.byref(lu)))
    try:
        b = rng.standard_normal((nblk, n)) + 1j * rng.standard_normal((nblk, n))
        db, dx = gade.DeviceArray.from_host(b.ravel()), gade.DeviceArray(nblk * n)
        gade.check(L.gade_blocklu_solve(lu, db.ptr, dx.ptr))
        x = dx.get().reshape(nblk, n)
    finally:
        L.gade_blocklu_destroy(lu)
    for q in range(3):
        want = np.linalg.solve(blocks[q], b[which == q].T).T
        got = x[which == q]
        assert np.all(np.abs(got - want).max(1) <= 1e-12 * np.abs(want).max(1)), (nblk, n, q)
