"""Passes of many sweeps (tl_deep*.hpp) against the one- and two-sweep passes
(TL_DEEP=0) on the same chunk.  A wave's strip is 108 to 120 columns wide in
FP64 and 232 to 248 in FP32, with ghosts of as many rows and columns as the
pass has sweeps: the meshes are narrower and wider than one and two strips,
ragged, and of fewer rows than the ghosts."""
import ctypes as C
import math

import numpy as np
import pytest

from helpers import interior
from tealeaf_ref_amd import _lib as L
from tealeaf_ref_amd.adjoint import chebyshev_coefs
from test_gpu_resident import SIZES as TILE_SIZES, _chunk, _norm_a, _start, env

pytestmark = pytest.mark.gpu

SIZES = [(3, 2), (7, 31), (107, 9), (109, 64), (217, 45), (250, 37), (501, 133), (130, 400)]


def _ppcg_sweeps(sizes, inner, reflective, envs, precond=1):
    """z after one outer iteration, i.e. the Chebyshev polynomial of r.

    Tolerance: with bounds that hold the spectrum the recurrence is stable, so
    a sweep's rounding (row sums of about 10 operations on terms of up to
    |A| |sd|, which is about 2 |r|) reaches z divided by theta = |A|/2 and is
    not amplified by more than the condition of the bounds used here, at most
    100.  That is 10 * 100 roundings per sweep relative to the largest z; and to
    the largest that enters, since alpha, whose sums are added in another order,
    is rounded there (many sweeps leave a z that is smaller by orders)."""
    pd = C.POINTER(C.c_double)
    for nx, ny in sizes:
        print(f"ppcg {nx}x{ny} inner {inner} reflective {reflective} {envs[1]}", flush=True)
        d, rx, ry = _chunk(nx, ny, precond, reflective)
        try:
            out = []
            for kw in envs:
                with env(**kw):
                    r0 = _start(d, rx, ry)
                    hi = 1.05 * _norm_a(d, rx, ry)
                    ca, cb, theta = chebyshev_coefs(hi / 100.0, hi, inner)
                    d.scalar("tl_cg_init")
                    L.call("tl_set_ppcg_active", 1)
                    d.scalar("tl_ppcg_init", 2)
                    # the switch to PPCG (tea_solve.f90:229-250)
                    L.call("tl_ppcg_init_sd", theta)
                    d.update_halo([0, 0, 0, 0, 0, 1, 1] + [0] * 4, 1)
                    L.call("tl_ppcg_inner", ca.ctypes.data_as(pd), cb.ctypes.data_as(pd), 1, inner)
                    L.call("tl_ppcg_update_z")
                    z0 = float(np.max(np.abs(interior(d.download("z"), 1))))
                    rro = d.scalar("tl_ppcg_init", 3)
                    st = L.LoopState(n_first=2, n_last=2, eps_abs=0.0, rro=rro, old_error=r0)
                    n = C.c_int(0)
                    rc = L.lib().tl_ppcg_loop(C.byref(st), ca.ctypes.data_as(pd),
                                              cb.ctypes.data_as(pd), inner, theta, C.byref(n))
                    L.call("tl_set_ppcg_active", 0)
                    out.append((rc, st.n_end, n.value, st.error, interior(d.download("z"), 1),
                                interior(d.download("p"), 1)))
        finally:
            d.close()
        ref, got = out
        assert got[:3] == ref[:3] == (L.TL_OK, 2, inner)
        tol = 1000.0 * inner * 2.0 ** -53
        for i in (4, 5):
            scale = max(z0, float(np.max(np.abs(ref[i]))))
            assert np.max(np.abs(got[i] - ref[i])) <= tol * scale, (nx, ny, i)


@pytest.mark.parametrize("inner", [4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 16, 21, 30])
@pytest.mark.parametrize("reflective", [False, True])
def test_ppcg_sweeps(inner, reflective):
    """Passes of many sweeps against passes of one and two."""
    _ppcg_sweeps(SIZES, inner, reflective, ({"TL_DEEP": 0}, {"TL_RESIDENT": 0}))


@pytest.mark.parametrize("rows,inner", [(1, 10), (2, 1), (3, 2), (4, 10), (6, 7), (0, 64)])
@pytest.mark.parametrize("reflective", [False, True])
def test_ppcg_on_chip(rows, inner, reflective):
    """The outer iterations on the chip against the passes of one and two sweeps."""
    _ppcg_sweeps(TILE_SIZES[1:], inner, reflective, ({"TL_DEEP": 0}, {"TL_RES_ROWS": rows}))


@pytest.mark.parametrize("precond,rows,inner", [(2, 1, 10), (2, 2, 3), (2, 3, 7), (2, 4, 10),
                                                (2, 6, 5), (3, 4, 10), (3, 4, 3)])
@pytest.mark.parametrize("reflective", [False, True])
def test_preconditioned_ppcg_on_chip(precond, rows, inner, reflective):
    """With jac_diag and jac_block against the passes of one and two sweeps; M^-1
    is at most 1, since A's diagonal and its blocks' eigenvalues are at least 1."""
    _ppcg_sweeps(TILE_SIZES[1:], inner, reflective, ({"TL_RESIDENT": 0}, {"TL_RES_ROWS": rows}),
                 precond)


@pytest.mark.parametrize("inner", [7, 10, 14])
@pytest.mark.parametrize("outers", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("way", [{"TL_RESIDENT": 0}, {"TL_RESIDENT": 1},
                                 {"TL_RES_ROWS": 2, "TL_RES_CHUNK": 2}])
def test_ppcg_outer_iterations(inner, outers, way):
    """Fields after 1 to 8 outer iterations, in which r and r_store change
    places every time, and the directions and u's updates go round 3 or 4; and
    on the chip, in one launch and in several.

    Tolerance: an outer iteration's rounding (test_ppcg_sweeps, through z) is
    carried on by CG's recurrences; 100 times the sum over the iterations, the
    condition of the bounds, relative to the largest r or u at the start, is
    1.3e-9 at most."""
    pd = C.POINTER(C.c_double)
    for nx, ny in ((7, 31), (109, 64), (250, 37)):
        print(f"deep ppcg outer {nx}x{ny} inner {inner} outers {outers}", flush=True)
        d, rx, ry = _chunk(nx, ny, 1, False)
        try:
            out = []
            for kw in ({"TL_DEEP": 0}, way):
                with env(**kw):
                    r0 = _start(d, rx, ry)
                    scale = {"r": float(np.max(np.abs(interior(d.download("r"), 1)))),
                             "u": float(np.max(np.abs(interior(d.download("u"), 1))))}
                    hi = 1.05 * _norm_a(d, rx, ry)
                    ca, cb, theta = chebyshev_coefs(hi / 100.0, hi, inner)
                    d.scalar("tl_cg_init")
                    L.call("tl_set_ppcg_active", 1)
                    d.scalar("tl_ppcg_init", 2)
                    L.call("tl_ppcg_init_sd", theta)
                    d.update_halo([0, 0, 0, 0, 0, 1, 1] + [0] * 4, 1)
                    L.call("tl_ppcg_inner", ca.ctypes.data_as(pd), cb.ctypes.data_as(pd), 1, inner)
                    L.call("tl_ppcg_update_z")
                    rro = d.scalar("tl_ppcg_init", 3)
                    st = L.LoopState(n_first=2, n_last=1 + outers, eps_abs=0.0, rro=rro,
                                     old_error=r0)
                    n = C.c_int(0)
                    rc = L.lib().tl_ppcg_loop(C.byref(st), ca.ctypes.data_as(pd),
                                              cb.ctypes.data_as(pd), inner, theta, C.byref(n))
                    L.call("tl_set_ppcg_active", 0)
                    out.append((rc, st.n_end, n.value,
                                {f: interior(d.download(f), 1) for f in ("u", "r", "r_store", "z",
                                                                         "p")}))
        finally:
            d.close()
        ref, got = out
        assert got[:3] == ref[:3] == (L.TL_OK, 1 + outers, inner * outers)
        tol = 100.0 * outers * 1000.0 * inner * 2.0 ** -53
        for f in ("u", "r", "r_store", "z", "p"):
            err = np.max(np.abs(got[3][f] - ref[3][f]))
            assert err <= tol * scale["u" if f == "u" else "r"], (nx, ny, f)


@pytest.mark.parametrize("inner", [4, 7, 10, 13, 20])
@pytest.mark.parametrize("rows", [None, 1, 4, 8, 12])
def test_mixed_sweeps(inner, rows):
    """The FP32 passes (rows None) and the on-chip loop inside the refined solver: all reach the true
    residual asked for, and |u - x| <= |u0 - A u| (the smallest eigenvalue of A
    is 1) bounds how far apart the two solutions may be."""
    for nx, ny in ((7, 31), (231, 40), (233, 64), (500, 133)):
        print(f"deep mixed {nx}x{ny} inner {inner}", flush=True)
        d, rx, ry = _chunk(nx, ny, 1, False)
        try:
            us = []
            for kw in ({"TL_DEEP": 0},
                       {"TL_RESIDENT": 0} if rows is None else {"TL_RES_ROWS": rows}):
                with env(**kw):
                    r0 = math.sqrt(_start(d, rx, ry))
                    st = d.mixed_solve(solver=L.MIXED_PPCG, rel_tol=1e-10, inner_steps=inner,
                                       presteps=20)
                    assert st.reason == L.LOOP_CONVERGED
                    us.append(interior(d.download("u"), 1))
        finally:
            d.close()
        assert np.linalg.norm(us[1] - us[0]) <= 2e-10 * r0 * 1.01


def _cheby(sizes, count, envs):
    """u, p, w and r after `count` iterations, and u's halo ring, which no way
    of running them changes, under two environments.

    Tolerance as in test_ppcg_sweeps, relative to the largest u and p; w and r
    hold u's rounding times |A|."""
    pd = C.POINTER(C.c_double)
    for nx, ny in sizes:
        print(f"chebyshev {nx}x{ny} count {count} {envs[1]}", flush=True)
        d, rx, ry = _chunk(nx, ny, 1, False)
        try:
            out = []
            for kw in envs:
                with env(**kw):
                    _start(d, rx, ry)
                    hi = 1.05 * _norm_a(d, rx, ry)
                    ca, cb, theta = chebyshev_coefs(hi / 100.0, hi, count + 1)
                    u = d.download("u")
                    u[0], u[-1], u[:, 0], u[:, -1] = 3.0, 4.0, 5.0, 6.0
                    d.upload("u", u)
                    L.call("tl_cheby_init", theta)
                    norm = C.c_double()
                    L.call("tl_cheby_run", ca.ctypes.data_as(pd), cb.ctypes.data_as(pd), 1, count,
                           1, C.byref(norm))
                    out.append([interior(d.download(f), 1) for f in ("u", "p", "w", "r")] +
                               [math.sqrt(norm.value), d.download("u")])
            norm_a = hi / 1.05
        finally:
            d.close()
        ref, got = out
        tol = 1000.0 * count * 2.0 ** -53
        big = float(np.max(np.abs(ref[0])))
        for i, scale in ((0, big), (1, big), (2, big * norm_a), (3, big * norm_a)):
            assert np.max(np.abs(got[i] - ref[i])) <= tol * scale, (nx, ny, i)
        assert abs(got[4] - ref[4]) <= tol * big * norm_a * math.sqrt(nx * ny)
        ring = np.ones(ref[5].shape, bool)
        ring[1:-1, 1:-1] = False
        ring[0, [0, -1]] = ring[-1, [0, -1]] = False  # corners are not carried
        assert np.array_equal(got[5][ring], ref[5][ring])


@pytest.mark.parametrize("count", [2, 3, 4, 5, 6, 8, 9, 10, 12, 17, 24, 31])
def test_cheby_iterations(count):
    """Passes of many iterations against passes of one and two."""
    _cheby(SIZES, count, ({"TL_DEEP": 0}, {"TL_RESIDENT": 0}))


@pytest.mark.parametrize("rows,count", [(1, 2), (2, 3), (3, 10), (4, 128), (6, 129), (8, 41),
                                        (0, 300)])
def test_cheby_on_chip(rows, count):
    """The whole run on the chip (128 iterations a launch) against the passes."""
    _cheby(TILE_SIZES[1:], count, ({"TL_RESIDENT": 0}, {"TL_RES_ROWS": rows}))
