"""A cooperative launch that is refused in the middle of a loop (another process has
come to hold the device's): the passes go on from the fields, scalars and histories
that the launches before it left, and the loop ends as one that ran in one way.
TL_RES_CHUNK makes several launches of a loop, TL_RES_REFUSE refuses one.

Tolerances: the iterations' arithmetic differs between the chip and the passes by
rounding only.  CG and PPCG solve to EPS, where two solutions differ by at most
2 EPS |r0| (the smallest eigenvalue of A is 1; sqrt|A| more with a preconditioner,
whose exit test is on sqrt(r.z)) and the drift that test_gpu_resident.py derives;
Jacobi's and Chebyshev's fields after a number of iterations as in
test_gpu_resident.py and test_gpu_deep.py."""
import ctypes as C
import math

import numpy as np
import pytest

from helpers import interior
from tealeaf_ref_amd import _lib as L
from tealeaf_ref_amd.adjoint import chebyshev_coefs
from test_gpu_resident import EPS, _chunk, _drift, _errors, _norm_a, _start, env

pytestmark = pytest.mark.gpu
PD = C.POINTER(C.c_double)
NX, NY = 300, 217


def _dp(a):
    return a.ctypes.data_as(PD)


def _fresh(precond):
    """A new chunk: a refusal lasts for the chunk's life."""
    return _chunk(NX, NY, precond, False)


@pytest.mark.parametrize("refuse", [0, 1, 3])
@pytest.mark.parametrize("precond", [1, 2, 3])
def test_cg(precond, refuse):
    out = []
    for kw in ({"TL_RESIDENT": 0}, {"TL_RES_CHUNK": 5, "TL_RES_REFUSE": refuse}):
        d, rx, ry = _fresh(precond)
        try:
            with env(**kw):
                r0 = _start(d, rx, ry)
                st = L.LoopState(n_first=1, n_last=4000, eps_abs=EPS * math.sqrt(r0),
                                 rro=d.scalar("tl_cg_init"), old_error=r0)
                al, be = np.zeros(4002), np.zeros(4002)
                assert L.lib().tl_cg_loop(C.byref(st), _dp(al), _dp(be)) == L.TL_OK
                norm_a = _norm_a(d, rx, ry)
                out.append((st, al, be, _errors(st.n_end), interior(d.download("u"), 1)))
        finally:
            d.close()
    (st0, al0, be0, er0, u0), (st1, al1, be1, er1, u1) = out
    assert st0.reason == st1.reason == L.LOOP_CONVERGED and st1.n_first == 1
    assert st0.n_end > 25 and abs(st1.n_end - st0.n_end) <= max(2, st0.n_end // 50)
    bound = 2 * EPS * math.sqrt(r0) * math.sqrt(norm_a if precond > 1 else 1.0)
    assert np.linalg.norm(u1 - u0) <= bound + 2 * _drift(st0.n_end, norm_a, u0)
    # the histories have no gap where the passes took over: the first 20
    # iterations' scalars agree to the drift of as many iterations
    for a, b in ((al0, al1), (be0, be1)):
        assert np.all(np.abs(a[1:21] - b[1:21]) <= 1e-9 * np.abs(a[1:21]))
        assert np.all(b[1:st1.n_end] != 0.0)
    assert np.all(np.abs(er0[:20] - er1[:20]) <= 1e-9 * er0[:20])
    assert er1[-1] == st1.error


@pytest.mark.parametrize("refuse", [0, 1, 2])
@pytest.mark.parametrize("precond", [1, 2, 3])
@pytest.mark.parametrize("inner", [4, 10])
def test_ppcg(precond, refuse, inner):
    out = []
    for kw in ({"TL_RESIDENT": 0}, {"TL_RES_CHUNK": 2, "TL_RES_REFUSE": refuse}):
        d, rx, ry = _fresh(precond)
        try:
            with env(**kw):
                r0 = _start(d, rx, ry)
                norm_a = _norm_a(d, rx, ry)
                ca, cb, theta = chebyshev_coefs(1.05 * norm_a / 100.0, 1.05 * norm_a, inner)
                d.scalar("tl_cg_init")
                L.call("tl_set_ppcg_active", 1)
                d.scalar("tl_ppcg_init", 2)
                L.call("tl_ppcg_init_sd", theta)
                L.call("tl_ppcg_inner", _dp(ca), _dp(cb), 1, inner)
                L.call("tl_ppcg_update_z")
                st = L.LoopState(n_first=2, n_last=8, eps_abs=0.0,
                                 rro=d.scalar("tl_ppcg_init", 3), old_error=r0)
                n = C.c_int(0)
                assert L.lib().tl_ppcg_loop(C.byref(st), _dp(ca), _dp(cb), inner, theta,
                                            C.byref(n)) == L.TL_OK
                L.call("tl_set_ppcg_active", 0)
                out.append((st.n_end, n.value, st.reason,
                            {f: interior(d.download(f), 1) for f in ("u", "r", "r_store", "z",
                                                                     "p")}))
        finally:
            d.close()
    (e0, n0, q0, f0), (e1, n1, q1, f1) = out
    assert (e0, n0, q0) == (e1, n1, q1) == (8, 7 * inner, L.LOOP_MAXITERS)
    # as test_ppcg_outer_iterations
    tol = 100.0 * 7 * 1000.0 * inner * 2.0 ** -53
    scale = {"u": np.max(np.abs(f0["u"])), "r": math.sqrt(r0)}
    for f in f0:
        assert np.max(np.abs(f1[f] - f0[f])) <= tol * scale["u" if f == "u" else "r"], f


@pytest.mark.parametrize("refuse", [0, 1, 2])
@pytest.mark.parametrize("pairs", [0, 1])
def test_jacobi(refuse, pairs):
    k, out = 37, []
    for kw in ({"TL_RESIDENT": 0}, {"TL_RES_CHUNK": 10, "TL_RES_REFUSE": refuse}):
        d, rx, ry = _fresh(1)
        try:
            with env(TL_SWEEP_PAIRS=pairs, **kw):
                _start(d, rx, ry)
                st = L.LoopState(n_first=1, n_last=k, eps_abs=0.0)
                assert L.lib().tl_jacobi_loop(C.byref(st)) == L.TL_OK
                assert (st.n_first, st.n_end, st.reason) == (1, k, L.LOOP_MAXITERS)
                out.append((_errors(k), interior(d.download("u"), 1)))
        finally:
            d.close()
    tol = 20.0 * k * 2.0 ** -53 * np.max(np.abs(out[0][1]))
    assert np.max(np.abs(out[0][1] - out[1][1])) <= tol
    assert np.max(np.abs(out[0][0] ** 2 - out[1][0] ** 2)) <= 2 * tol * NX * NY * 1.01


@pytest.mark.parametrize("count", [129, 300])
@pytest.mark.parametrize("refuse", [0, 1, 2])
@pytest.mark.parametrize("want_norm", [0, 1])
def test_chebyshev(count, refuse, want_norm):
    """128 iterations a launch: one to four remain, or some hundred."""
    out = []
    for kw in ({"TL_RESIDENT": 0}, {"TL_RES_REFUSE": refuse}):
        d, rx, ry = _fresh(1)
        try:
            with env(**kw):
                _start(d, rx, ry)
                norm_a = _norm_a(d, rx, ry)
                ca, cb, theta = chebyshev_coefs(1.05 * norm_a / 100.0, 1.05 * norm_a, count + 1)
                L.call("tl_cheby_init", theta)
                norm = C.c_double()
                L.call("tl_cheby_run", _dp(ca), _dp(cb), 1, count, want_norm, C.byref(norm))
                out.append([interior(d.download(f), 1) for f in ("u", "p", "w", "r")] +
                           [math.sqrt(norm.value)])
        finally:
            d.close()
    ref, got = out
    tol = 1000.0 * count * 2.0 ** -53
    big = float(np.max(np.abs(ref[0])))
    for i, scale in ((0, big), (1, big), (2, big * norm_a), (3, big * norm_a)):
        assert np.max(np.abs(got[i] - ref[i])) <= tol * scale, i
    if want_norm:
        assert abs(got[4] - ref[4]) <= tol * big * norm_a * math.sqrt(NX * NY)
