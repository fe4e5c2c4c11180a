"""tl_cg_loop while PPCG is active, without a preconditioner: p comes from z as
it is in memory, as tl_cg_calc_p has it there (tea_leaf_cg_kernel.f90's calc_p with
tl_ppcg_active), on every mesh, whichever kernels run."""
import ctypes as C

import numpy as np
import pytest

from helpers import interior
from tealeaf_ref_amd import _lib as L
from test_gpu_resident import _chunk, _start, env

pytestmark = pytest.mark.gpu


def _loop(d, rx, ry, iters, z, active):
    """p before and after `iters` iterations, u, r and the betas."""
    r0 = _start(d, rx, ry)
    rro = d.scalar("tl_cg_init")
    d.upload("z", z)
    p0 = interior(d.download("p"), 1)
    L.call("tl_set_ppcg_active", active)
    st = L.LoopState(n_first=1, n_last=iters, eps_abs=0.0, rro=rro, old_error=r0)
    be = np.zeros(iters + 2)
    rc = L.lib().tl_cg_loop(C.byref(st), None, be.ctypes.data_as(C.POINTER(C.c_double)))
    L.call("tl_set_ppcg_active", 0)
    assert rc == L.TL_OK and st.n_end == iters
    return p0, [interior(d.download(f), 1) for f in ("p", "u", "r")], be


@pytest.mark.parametrize("nx,ny", [(7, 31), (130, 70), (300, 517), (1500, 1600)])
def test_p_comes_from_z(nx, ny):
    """One iteration: p = z + beta p, of two operations, each rounded once; and the
    same bits with the on-chip loops off, as neither runs them."""
    rng = np.random.default_rng(5)
    z = rng.uniform(-1.0, 1.0, size=(ny + 2, nx + 2))
    d, rx, ry = _chunk(nx, ny, 1, False)
    try:
        p0, (p, u, r), be = _loop(d, rx, ry, 1, z, 1)
        zi = interior(z, 1)
        bound = 2 * 2.0 ** -53 * (np.abs(zi) + 2 * np.abs(be[1] * p0))
        assert np.all(np.abs(p - (zi + be[1] * p0)) <= bound)
        for iters in (1, 2, 5):
            got = _loop(d, rx, ry, iters, z, 1)[1]
            with env(TL_RESIDENT=0):
                ref = _loop(d, rx, ry, iters, z, 1)[1]
            assert all(np.array_equal(a, b) for a, b in zip(got, ref))
        # not active: from r
        p0, (p, u, r), be = _loop(d, rx, ry, 1, z, 0)
        bound = 2 * 2.0 ** -53 * (np.abs(r) + 2 * np.abs(be[1] * p0))
        assert np.all(np.abs(p - (r + be[1] * p0)) <= bound)
    finally:
        d.close()
