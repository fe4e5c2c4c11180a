"""The CG update pass that applies u += alpha p of four iterations together
(TL_CG_DEFER) against the one that applies it in each: the additions are the
same in the same order, so every field and scalar has the same bits, wherever
in the group of four the loop ends."""
import ctypes as C
import math

import numpy as np
import pytest

from helpers import interior
from tealeaf_ref_amd import _lib as L
from test_gpu_resident import _chunk, _start, env

pytestmark = pytest.mark.gpu


def _run(d, rx, ry, precond, n_last, eps, switch):
    r0 = _start(d, rx, ry)
    rro = d.scalar("tl_cg_init")
    st = L.LoopState(n_first=1, n_last=n_last, eps_abs=eps * math.sqrt(r0), rro=rro, old_error=r0,
                     check_switch=1 if switch else 0, epslim=math.inf, presteps=switch)
    pd = C.POINTER(C.c_double)
    al, be = np.zeros(n_last + 2), np.zeros(n_last + 2)
    rc = L.lib().tl_cg_loop(C.byref(st), al.ctypes.data_as(pd), be.ctypes.data_as(pd))
    names = ("u", "r", "p", "w") + (("z",) if precond > 1 else ())
    return ([rc, st.n_end, st.reason, st.rro, st.error, al, be] +
            [interior(d.download(f), 1) for f in names])


@pytest.mark.parametrize("precond", [1, 2, 3])
@pytest.mark.parametrize("nx,ny", [(130, 67), (513, 40)])
def test_same_bits(precond, nx, ny):
    cases = [(n, 0.0, 0) for n in (1, 2, 3, 4, 5, 7, 8, 18)]
    cases += [(400, 1e-6, 0), (60, 0.0, 6), (60, 0.0, 9)]
    d, rx, ry = _chunk(nx, ny, precond, False)
    try:
        for n_last, eps, switch in cases:
            print(f"cg defer {nx}x{ny} precond {precond} n_last {n_last} eps {eps} switch {switch}",
                  flush=True)
            out = []
            for on in (0, 1):
                with env(TL_RESIDENT=0, TL_CG_DEFER=on):
                    out.append(_run(d, rx, ry, precond, n_last, eps, switch))
            assert out[0][0] == L.TL_OK
            for a, b in zip(*out):
                assert np.array_equal(a, b)
    finally:
        d.close()
