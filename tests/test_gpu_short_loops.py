"""Loops of a few iterations: they take the kernels that are the faster there, not
those that pay off over many.  Both routes are timed in turn on the same chunk;
where the rule picks the older one the two are the same launches, so that their
times differ by noise only (a few per cent at 20 us and more), against 1.19
to 1.45 where the rule is missing; lower quartiles are compared, which a busy host
moves least."""
import ctypes as C
import time

import numpy as np
import pytest

from helpers import interior
from tealeaf_ref_amd import _lib as L
from tealeaf_ref_amd.adjoint import chebyshev_coefs
from test_gpu_deep import SIZES, _cheby
from test_gpu_resident import _chunk, _norm_a, _start, env

pytestmark = pytest.mark.gpu
MARGIN = 1.15


def _times(call, routes, repeats=41):
    """Lower quartile of the seconds of `call` under each environment, in turn."""
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
    return [float(np.percentile(t, 25)) for t in times]


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

        new, old = _times(call, ({}, {"TL_CG_DEFER": 0}))
        print(f"one cg iteration {new * 1e6:.1f} us, u in each update {old * 1e6:.1f}", flush=True)
        assert new <= MARGIN * old
    finally:
        d.close()


@pytest.mark.parametrize("n,count", [(512, 2), (512, 3), (2000, 2), (4096, 2), (4096, 3)])
def test_few_chebyshev_iterations(n, count):
    """Two or three iterations are left to the two-iteration passes, on meshes that
    fit the chip and beyond: the same fields to the bit, in the same time."""
    pd = C.POINTER(C.c_double)
    d, rx, ry = _chunk(n, n, 1, False)
    try:
        out = []
        _start(d, rx, ry)
        hi = 1.05 * _norm_a(d, rx, ry)
        ca, cb, theta = chebyshev_coefs(hi / 100.0, hi, count + 1)
        norm = C.c_double()

        def call():
            L.call("tl_cheby_run", ca.ctypes.data_as(pd), cb.ctypes.data_as(pd), 1, count, 1,
                   C.byref(norm))

        for kw in ({}, {"TL_DEEP": 0}):
            _start(d, rx, ry)
            L.call("tl_cheby_init", theta)
            with env(**kw):
                call()
            out.append([interior(d.download(f), 1) for f in ("u", "p", "r")])
        assert all(np.array_equal(a, b) for a, b in zip(*out))
        new, old = _times(call, ({}, {"TL_DEEP": 0}))
        print(f"chebyshev {n}^2 {count} its {new * 1e6:.1f} us, pairs {old * 1e6:.1f}", flush=True)
        assert new <= MARGIN * old
    finally:
        d.close()


@pytest.mark.parametrize("n,count", [(250, 4), (512, 5), (250, 8), (1024, 2), (1024, 8)])
def test_short_chebyshev_runs_leave_the_chip(n, count):
    """Under nine iterations the passes are the faster on a mesh of more than one
    block that fits the chip: the bits of the passes."""
    pd = C.POINTER(C.c_double)
    d, rx, ry = _chunk(n, n, 1, False)
    try:
        out = []
        for kw in ({}, {"TL_RESIDENT": 0}):
            _start(d, rx, ry)
            hi = 1.05 * _norm_a(d, rx, ry)
            ca, cb, theta = chebyshev_coefs(hi / 100.0, hi, count + 1)
            L.call("tl_cheby_init", theta)
            norm = C.c_double()
            with env(**kw):
                L.call("tl_cheby_run", ca.ctypes.data_as(pd), cb.ctypes.data_as(pd), 1, count, 1,
                       C.byref(norm))
            out.append([interior(d.download(f), 1) for f in ("u", "p", "r")] + [norm.value])
        assert all(np.array_equal(a, b) for a, b in zip(*out))
    finally:
        d.close()


@pytest.mark.parametrize("count", [2, 3])
def test_many_step_pass_of_two(count):
    """The many-step pass of two iterations, which meshes of 40 million cells and
    more take, against the two-iteration passes."""
    _cheby(SIZES, count, ({"TL_DEEP": 0}, {"TL_RESIDENT": 0, "TL_DEEP": 2}))
