"""The solver loops that keep the mesh on the chip (tl_resident.hip) against
the pass kernels (TL_RESIDENT=0) on the same chunk: tiles of 128 columns and
8 to 64 rows, so the sizes lie on, just below and just past those, with one
tile, one row or column of tiles, and both.

Bound: A = I + L with L positive semidefinite, so its smallest eigenvalue is 1
and the error of an iterate is at most its residual, |u - x| <= |u0 - A u|.
Two solves that stop at a recurrence residual of eps |r0| therefore differ by
at most 2 eps |r0| plus what the recurrence residual has drifted from the true
one, which for k iterations of CG is at most a small multiple of
k 2^-53 |A| max|u_i| (Greenbaum 1997); 10 is taken for the multiple, and |A| is
at most the largest row sum.  Neither bound depends on the order of the sums."""
import ctypes as C
import math
import os

import numpy as np
import pytest

from helpers import interior, random_chunk
from tealeaf_ref_amd import _lib as L

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (2, 9), (127, 8), (128, 64), (129, 65), (255, 33), (257, 130), (300, 517),
         (1030, 71), (1281, 700)]


class env:
    def __init__(self, **kw):
        self.kw = {k: str(v) for k, v in kw.items()}

    def __enter__(self):
        self.old = {k: os.environ.get(k) for k in self.kw}
        os.environ.update(self.kw)

    def __exit__(self, *a):
        for k, v in self.old.items():
            os.environ.pop(k, None) if v is None else os.environ.__setitem__(k, v)


def _chunk(nx, ny, precond, reflective, seed=7):
    rho, e1, vol, rx, ry = random_chunk(nx, ny, 1, seed)
    d = L.Device(nx, ny, 1)
    d.set_options(L.CONDUCTIVITY, precond, reflective)
    d.upload("density", rho)
    d.upload("energy1", e1)
    return d, rx, ry


def _start(d, rx, ry):
    d.update_halo([1, 0, 1] + [0] * 8, 1)
    d.common_init(rx, ry)
    d.update_halo([0, 0, 0, 1] + [0] * 7, 1)
    L.call("tl_calc_residual")
    return d.scalar("tl_calc_2norm", 1)


def _cg(d, rx, ry, n_last, eps=0.0):
    r0 = _start(d, rx, ry)
    rro = d.scalar("tl_cg_init")
    st = L.LoopState(n_first=1, n_last=n_last, eps_abs=eps * math.sqrt(r0), rro=rro, old_error=r0)
    rc = L.lib().tl_cg_loop(C.byref(st), None, None)
    return st, rc


def _norm_a(d, rx, ry):
    """Largest row sum of |A| (1 + twice the face coefficients of a cell)."""
    kx, ky = d.download("kx"), d.download("ky")
    k = rx * (kx[1:-1, 1:-1] + kx[1:-1, 2:]) + ry * (ky[1:-1, 1:-1] + ky[2:, 1:-1])
    return 1.0 + 2.0 * float(np.max(k))


EPS = 1e-10


def _drift(k, norm_a, u):
    return 10.0 * k * 2.0 ** -53 * norm_a * float(np.linalg.norm(u))


def _cont(d, st, n_last, r0):
    """Go on with the loop that stopped in `st`."""
    st2 = L.LoopState(n_first=st.n_end + 1, n_last=n_last, eps_abs=EPS * math.sqrt(r0),
                      rro=st.rro, old_error=st.error)
    assert L.lib().tl_cg_loop(C.byref(st2), None, None) == L.TL_OK
    return st2


@pytest.mark.parametrize("rows", [0, 1, 2, 3, 4, 6, 8])
@pytest.mark.parametrize("precond,reflective", [(1, False), (1, True), (2, False), (2, True),
                                                (3, False), (3, True)])
def test_cg_matches_passes(precond, reflective, rows):
    """Both solve to EPS; and the fields the chip leaves after a few
    iterations (u, r, p, z) are those the pass kernels go on from."""
    for nx, ny in SIZES:
        if (nx, ny) == (1, 1):
            continue  # its residual is zero: nothing to iterate on
        print(f"resident cg {nx}x{ny} precond {precond} refl {reflective} rows {rows}", flush=True)
        d, rx, ry = _chunk(nx, ny, precond, reflective)
        try:
            with env(TL_RESIDENT=0):
                st0, rc0 = _cg(d, rx, ry, 4000, EPS)
                u_pass = interior(d.download("u"), 1)
            with env(TL_RES_ROWS=rows):
                st1, rc1 = _cg(d, rx, ry, 4000, EPS)
                u_res = interior(d.download("u"), 1)
                r_res = interior(d.download("r"), 1)
                d.update_halo([0, 0, 0, 1] + [0] * 7, 1)  # tl_calc_residual reads u's halo
                L.call("tl_calc_residual")
                r_true = interior(d.download("r"), 1)
                r0 = _start(d, rx, ry)
                st2, rc2 = _cg(d, rx, ry, max(1, st1.n_end // 2), EPS)
            with env(TL_RESIDENT=0):
                st3 = _cont(d, st2, 4000, r0)
                u_cont = interior(d.download("u"), 1)
            norm_a = _norm_a(d, rx, ry)
        finally:
            d.close()
        assert (rc0, rc1, rc2) == (L.TL_OK,) * 3
        assert st0.reason == st1.reason == st3.reason == L.LOOP_CONVERGED
        # rounding moves an exit by an iteration or two, never by a share of them
        for st in (st1, st3):
            assert abs(st.n_end - st0.n_end) <= max(2, st0.n_end // 50), (st0.n_end, st.n_end)
        drift = _drift(st0.n_end, norm_a, u_pass)
        bound = 2 * EPS * math.sqrt(r0) + 2 * drift
        if precond > 1:
            # the exit test is on sqrt(r.z) there, and |r|^2 <= |M| r.z with
            # |M| the largest diagonal (or 4-row block) entry sum, at most |A|
            bound = 2 * EPS * math.sqrt(r0) * math.sqrt(norm_a) + 2 * drift
        assert np.linalg.norm(u_res - u_pass) <= bound
        assert np.linalg.norm(u_cont - u_pass) <= bound
        assert np.linalg.norm(r_res - r_true) <= 2 * drift


def test_cg_in_several_launches():
    """A loop that comes back to the host between launches goes on as if it
    had not: the same kernel on the same fields, bit for bit."""
    d, rx, ry = _chunk(200, 150, 1, False)
    try:
        st0, _ = _cg(d, rx, ry, 300, eps=1e-9)
        u0 = d.download("u")
        with env(TL_RES_CHUNK=7):
            st1, _ = _cg(d, rx, ry, 300, eps=1e-9)
        u1 = d.download("u")
    finally:
        d.close()
    assert st0.reason == L.LOOP_CONVERGED and st0.n_end > 14
    assert (st1.n_end, st1.reason, st1.error) == (st0.n_end, st0.reason, st0.error)
    assert np.array_equal(u1, u0)


def _errors(k):
    """Exit-test errors of iterations 1..k (the library's array starts at 0)."""
    err = np.zeros(k + 1)
    L.call("tl_loop_errors", 1, k, err.ctypes.data_as(C.POINTER(C.c_double)))
    return err[1:]


def _jacobi(u, u0, kx, ky, rx, ry, k):
    """k iterations of tea_leaf_jacobi_kernel.f90:60-66, in its order of
    operations, reading zero outside the mesh."""
    c = (slice(1, -1), slice(1, -1))
    kl, kr, kd, ku = kx[c], kx[1:-1, 2:], ky[c], ky[2:, 1:-1]
    un = np.zeros_like(u)
    un[c] = u[c]
    for _ in range(k):
        v = ((u0[c] + rx * (kr * un[1:-1, 2:] + kl * un[1:-1, :-2]) +
              ry * (ku * un[2:, 1:-1] + kd * un[:-2, 1:-1])) /
             (1.0 + rx * (kl + kr) + ry * (kd + ku)))
        un[c] = v
    return un[c]


@pytest.mark.parametrize("rows", [0, 1, 2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("reflective", [False, True])
def test_jacobi_matches_passes(reflective, rows):
    """u after a number of Jacobi iterations, in one launch and in several.

    Tolerance: an iteration's rounding is at most 10 operations' on terms of at
    most the largest u, and an iteration never increases the largest
    difference of two iterates (its row sums are below 1), so after k
    iterations the two differ by at most 2 * 10 k 2^-53 max|u|.  The sum of |u -
    un| then differs by at most twice that per cell, besides its own rounding.
    The iterates on the chip are the reference's to the bit."""
    k = 37
    for nx, ny in SIZES[1:]:  # 1x1 has converged before the first iteration
        print(f"resident jacobi {nx}x{ny} refl {reflective} rows {rows}", flush=True)
        d, rx, ry = _chunk(nx, ny, 1, reflective)
        try:
            out = []
            for kw in ({"TL_RESIDENT": 0}, {"TL_RES_ROWS": rows},
                       {"TL_RES_ROWS": rows, "TL_RES_CHUNK": 10}):
                with env(**kw):
                    _start(d, rx, ry)
                    exact = [d.download(f) for f in ("u", "u0", "kx", "ky")]
                    st = L.LoopState(n_first=1, n_last=k, eps_abs=0.0)
                    assert L.lib().tl_jacobi_loop(C.byref(st)) == L.TL_OK
                    out.append((st.n_end, st.reason, _errors(k), interior(d.download("u"), 1)))
        finally:
            d.close()
        ref = out[0]
        big = float(np.max(np.abs(ref[3])))
        tol = 20.0 * k * 2.0 ** -53 * big
        for got in out[1:]:
            assert got[:2] == ref[:2] == (k, L.LOOP_MAXITERS)
            assert np.max(np.abs(got[3] - ref[3])) <= tol
            assert np.max(np.abs(got[2] ** 2 - ref[2] ** 2)) <= 2 * tol * nx * ny * 1.01
        assert np.array_equal(out[1][3], out[2][3])
        assert np.array_equal(out[1][3], _jacobi(*exact, rx, ry, k))


def test_jacobi_exit():
    """The exit test of an iteration ends the loop there."""
    d, rx, ry = _chunk(300, 200, 1, False)
    try:
        out = []
        for resident in (0, 1):
            with env(TL_RESIDENT=resident):
                _start(d, rx, ry)
                st = L.LoopState(n_first=1, n_last=60, eps_abs=0.0)
                assert L.lib().tl_jacobi_loop(C.byref(st)) == L.TL_OK
                err = _errors(60)
                for n in (1, 8, 41):  # a bound between the errors of n - 1 and n
                    eps = 2.0 * err[0] if n == 1 else 0.5 * (err[n - 2] + err[n - 1])
                    _start(d, rx, ry)
                    st = L.LoopState(n_first=1, n_last=60, eps_abs=eps)
                    assert L.lib().tl_jacobi_loop(C.byref(st)) == L.TL_OK
                    out.append((st.n_end, st.reason))
                assert out[-3:] == [(n, L.LOOP_CONVERGED) for n in (1, 8, 41)]
    finally:
        d.close()
    assert out[:3] == out[3:]


def test_wait_that_runs_out_is_an_error():
    """Every wait of the launch is made to run out (a negative limit): all
    blocks leave the kernel, the call fails, and the next one runs."""
    d, rx, ry = _chunk(300, 200, 1, False)
    try:
        ref, rc = _cg(d, rx, ry, 20)
        assert rc == L.TL_OK
        with env(TL_RES_LIMIT=-1, TL_RES_ROWS=4):
            _, rc = _cg(d, rx, ry, 20)
            assert rc == L.ERR_HIP
            assert b"waited too long" in L.lib().tl_last_error()
        st, rc = _cg(d, rx, ry, 20)
        assert rc == L.TL_OK and (st.n_end, st.error) == (ref.n_end, ref.error)
    finally:
        d.close()
