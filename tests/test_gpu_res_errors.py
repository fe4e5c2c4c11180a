"""Waits of the on-chip loops that run out: every wait of a launch is made to (a
negative limit), all blocks leave the kernel, and the call that launched it
fails, whether or not it returns a scalar; the next one runs."""
import ctypes as C

import numpy as np
import pytest

from helpers import interior
from tealeaf_ref_amd import _lib as L
from tealeaf_ref_amd.adjoint import chebyshev_coefs
from test_gpu_resident import _chunk, _norm_a, _start, env

pytestmark = pytest.mark.gpu
PD = C.POINTER(C.c_double)


def _dp(a):
    return a.ctypes.data_as(PD)


def _cheby(d, rx, ry, count, want_norm, limit):
    """Return code and message of a run of `count` iterations, and u."""
    _start(d, rx, ry)
    hi = 1.05 * _norm_a(d, rx, ry)
    ca, cb, theta = chebyshev_coefs(hi / 100.0, hi, count + 1)
    L.call("tl_cheby_init", theta)
    norm = C.c_double()
    with env(**limit):
        rc = L.lib().tl_cheby_run(_dp(ca), _dp(cb), 1, count, want_norm, C.byref(norm))
        message = L.lib().tl_last_error()
    return rc, message, interior(d.download("u"), 1)


@pytest.mark.parametrize("want_norm", [0, 1])
@pytest.mark.parametrize("count", [20, 300])
def test_chebyshev(count, want_norm):
    """One launch and three; the fields after a run without limit are the same
    whether or not the norm was asked for (the same kernel on the same fields)."""
    d, rx, ry = _chunk(300, 200, 1, False)
    try:
        rc, message, _ = _cheby(d, rx, ry, count, want_norm, {"TL_RES_LIMIT": -1})
        assert rc == L.ERR_HIP and b"waited too long" in message
        rc, _, u0 = _cheby(d, rx, ry, count, want_norm, {})
        assert rc == L.TL_OK
        rc, _, u1 = _cheby(d, rx, ry, count, 1 - want_norm, {})
        assert rc == L.TL_OK and np.array_equal(u0, u1)
    finally:
        d.close()


def test_jacobi():
    d, rx, ry = _chunk(300, 200, 1, False)
    try:
        for limit, want in (({"TL_RES_LIMIT": -1}, L.ERR_HIP), ({}, L.TL_OK)):
            _start(d, rx, ry)
            st = L.LoopState(n_first=1, n_last=10, eps_abs=0.0)
            with env(**limit):
                assert L.lib().tl_jacobi_loop(C.byref(st)) == want
    finally:
        d.close()


def test_ppcg():
    d, rx, ry = _chunk(300, 200, 1, False)
    try:
        for limit, want in (({"TL_RES_LIMIT": -1}, L.ERR_HIP), ({}, L.TL_OK)):
            r0 = _start(d, rx, ry)
            hi = 1.05 * _norm_a(d, rx, ry)
            ca, cb, theta = chebyshev_coefs(hi / 100.0, hi, 10)
            d.scalar("tl_cg_init")
            L.call("tl_set_ppcg_active", 1)
            d.scalar("tl_ppcg_init", 2)
            L.call("tl_ppcg_init_sd", theta)
            L.call("tl_ppcg_inner", _dp(ca), _dp(cb), 1, 10)
            L.call("tl_ppcg_update_z")
            rro = d.scalar("tl_ppcg_init", 3)
            st = L.LoopState(n_first=2, n_last=4, eps_abs=0.0, rro=rro, old_error=r0)
            n = C.c_int(0)
            with env(**limit):
                assert L.lib().tl_ppcg_loop(C.byref(st), _dp(ca), _dp(cb), 10, theta,
                                            C.byref(n)) == want
            L.call("tl_set_ppcg_active", 0)
    finally:
        d.close()
