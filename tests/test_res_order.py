"""The exchanges of the on-chip loops (tl_resident.hpp): no word of the buffers
is written again before its readers have it, whichever block or wave lags."""
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

from helpers import interior
from tealeaf_ref_amd import _lib as L
from tealeaf_ref_amd.adjoint import chebyshev_coefs
from test_gpu_resident import _chunk, _norm_a, _start, env

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "tealeaf_ref_amd", "csrc")


def test_no_schedule_ends_stuck(tmp_path):
    """A model of the exchanges with the rule of tl_res_order.hpp: CG, Jacobi,
    Chebyshev, and PPCG with odd and even inner steps, in each of which one block
    or one of its waves moves only when nothing else can.  The model does end
    stuck where sums take the copy of their exchange's number: with odd inner
    steps, on grids whose blocks are further apart than those."""
    exe = str(tmp_path / "model")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(HERE, "res_order_model.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True, timeout=300).stdout
    rows = re.findall(r"(\w+) (\w+) (\d+)x(\d+) runs (\d+) stuck (\d+)", out)
    assert len(rows) == 2 * 11 * 6
    for rule, loop, tx, ty, runs, stuck in rows:
        if rule == "sums":
            assert int(runs) > 0 and int(stuck) == 0, (loop, tx, ty)
        elif loop in ("ppcg1", "ppcg3", "ppcg5", "ppcg7", "ppcg9"):
            if int(tx) + int(ty) - 2 > int(loop[4:]):
                assert int(stuck) > 0, (loop, tx, ty)
        else:
            assert int(stuck) == 0, (loop, tx, ty)


MANY_TILES = [(1, 1, 100, 2001), (1, 2, 900, 900), (2, 1, 100, 1500), (3, 4, 70, 4000)]


@pytest.mark.gpu
# with a preconditioner one or two inner steps run per routine
@pytest.mark.parametrize("precond,rows,nx,ny,inner", [
    (*m, inner) for m in MANY_TILES for inner in (1, 2, 3, 5, 7, 9) if m[0] == 1 or inner > 2])
def test_ppcg_many_tiles(inner, precond, rows, nx, ny):
    """Several outer iterations on the chip, on grids of up to 251 tiles in a column
    and of 8 by 57, against the passes.

    Tolerance: an outer iteration's rounding is that of its sweeps, 10 * 100
    roundings each with bounds of condition 100 (row sums of about 10 operations),
    which CG's recurrences carry on with at most the condition again: 100 times
    the sum over the iterations, relative to the largest u or r at the start."""
    pd = C.POINTER(C.c_double)
    outers = 6
    print(f"ppcg many tiles {nx}x{ny} precond {precond} inner {inner}", flush=True)
    d, rx, ry = _chunk(nx, ny, precond, False)
    try:
        out = []
        for kw in ({"TL_RESIDENT": 0}, {"TL_RES_ROWS": rows}):
            with env(**kw):
                r0 = _start(d, rx, ry)
                scale = {f: float(np.max(np.abs(interior(d.download(f), 1)))) for f in ("u", "r")}
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
                st = L.LoopState(n_first=2, n_last=1 + outers, eps_abs=0.0, rro=rro, old_error=r0)
                n = C.c_int(0)
                rc = L.lib().tl_ppcg_loop(C.byref(st), ca.ctypes.data_as(pd),
                                          cb.ctypes.data_as(pd), inner, theta, C.byref(n))
                L.call("tl_set_ppcg_active", 0)
                out.append((rc, st.n_end, n.value,
                            {f: interior(d.download(f), 1) for f in ("u", "r", "z", "p")}))
    finally:
        d.close()
    ref, got = out
    assert got[:3] == ref[:3] == (L.TL_OK, 1 + outers, inner * outers)
    tol = 100.0 * outers * 1000.0 * inner * 2.0 ** -53
    for f in ("u", "r", "z", "p"):
        err = np.max(np.abs(got[3][f] - ref[3][f]))
        assert err <= tol * scale["u" if f == "u" else "r"], f
