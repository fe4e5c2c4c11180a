"""Loops of a few iterations: they take the kernels that are the faster there, not
those that pay off over many.  Both routes are timed in turn on the same chunk;
where the rule picks the older one the two are the same launches, so that their
medians differ by noise only (a few per cent at 20 us and more), against 1.19
to 1.45 where the rule is missing."""
import ctypes as C
import time

import numpy as np
import pytest

from tealeaf_ref_amd import _lib as L
from test_gpu_resident import _chunk, _start, env

pytestmark = pytest.mark.gpu
MARGIN = 1.12


def _medians(call, routes, repeats=31):
    """Median seconds of `call` under each environment, in turn."""
    times = [[] for _ in routes]
    for k in range(repeats + 3):
        for t, kw in zip(times, routes):
            with env(**kw):
                L.call("tl_synchronize")
                a = time.perf_counter()
                call()
                L.call("tl_synchronize")
                if k >= 3:
                    t.append(time.perf_counter() - a)
    return [float(np.median(t)) for t in times]


def test_one_cg_iteration():
    """u's update is not put off in a loop of one iteration (PPCG's later steps run
    such a one before the switch)."""
    d, rx, ry = _chunk(3000, 3000, 1, False)
    try:
        r0 = _start(d, rx, ry)
        st = L.LoopState(n_first=1, n_last=1, eps_abs=0.0, rro=d.scalar("tl_cg_init"), old_error=r0)

        def call():
            st.n_first = st.n_last = 1
            assert L.lib().tl_cg_loop(C.byref(st), None, None) == L.TL_OK

        new, old = _medians(call, ({}, {"TL_CG_DEFER": 0}))
        print(f"one cg iteration {new * 1e6:.1f} us, u in each update {old * 1e6:.1f}", flush=True)
        assert new <= MARGIN * old
    finally:
        d.close()
