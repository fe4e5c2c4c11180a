"""The w pass with faces formed from the density (k_loop_w, DENS) against the
same pass reading Kx and Ky (TL_DENS_FACES=0), on meshes within and beyond a
wave (128 columns), a block's tile (512) and ragged against both."""
import ctypes as C
import math

import numpy as np
import pytest

from helpers import interior
from tealeaf_ref_amd import _lib as L
from test_gpu_resident import _chunk, _norm_a, _start, env

pytestmark = pytest.mark.gpu

SIZES = [(1, 9), (2, 5), (127, 8), (129, 33), (512, 40), (515, 61), (1030, 7)]
FIELDS = ("u", "r", "p", "w")


def _cg(d, rx, ry, its, before=None):
    r0 = _start(d, rx, ry)
    if before:
        before()
    rro = d.scalar("tl_cg_init")
    st = L.LoopState(n_first=1, n_last=its, eps_abs=0.0, rro=rro, old_error=r0)
    assert L.lib().tl_cg_loop(C.byref(st), None, None) == L.TL_OK
    return {f: interior(d.download(f), 1) for f in FIELDS}


@pytest.mark.parametrize("coefficient", [L.CONDUCTIVITY, L.RECIP_CONDUCTIVITY])
@pytest.mark.parametrize("reflective", [False, True])
def test_same_faces(coefficient, reflective):
    """The faces are the same to the bit, but not the products that the compiler
    fuses in w; and with reflective faces those on the mesh's edge, whose two
    terms cancel, are left out.  The rounding of w = A p's terms, at most 2^-52
    |A| max|p| an iteration, is carried on by CG as in its rounding bounds, 100
    times at most here; p and r are at most |A| max|u|."""
    its = 9
    for nx, ny in SIZES:
        print(f"density faces {nx}x{ny} coefficient {coefficient} refl {reflective}", flush=True)
        d, rx, ry = _chunk(nx, ny, 1, reflective)
        d.set_options(coefficient, 1, reflective)
        try:
            with env(TL_RESIDENT=0, TL_DENS_FACES=0):
                ref = _cg(d, rx, ry, its)
            with env(TL_RESIDENT=0, TL_DENS_FACES=1):
                got = _cg(d, rx, ry, its)
            norm_a = _norm_a(d, rx, ry)
            scale = {f: norm_a * float(np.max(np.abs(ref["u"]))) for f in FIELDS}
            scale["w"] = norm_a * max(scale["p"], float(np.max(np.abs(ref["p"]))))
        finally:
            d.close()
        for f in FIELDS:
            err = np.max(np.abs(got[f] - ref[f]))
            print(f"  {f} {err / (its * 2.0 ** -52 * scale[f]):.2g}", flush=True)
            assert err <= 100 * its * 2.0 ** -52 * scale[f], (nx, ny, f)


@pytest.mark.parametrize("field", ["kx", "density"])
def test_faces_written_by_the_caller(field):
    """A call that writes the faces or the density after they were formed: the
    loop takes Kx and Ky as they are."""
    nx, ny = 300, 41
    d, rx, ry = _chunk(nx, ny, 1, False)
    try:
        out = []
        for dens in (0, 1):
            with env(TL_RESIDENT=0, TL_DENS_FACES=dens):
                d.upload("density", d.download("density"))

                def before():
                    v = d.download(field)
                    v[1:-1, 2:-1] *= 0.5
                    d.upload(field, v)

                rho = d.download("density")
                out.append(_cg(d, rx, ry, 7, before))
                d.upload("density", rho)
    finally:
        d.close()
    for f in FIELDS:
        assert np.array_equal(out[0][f], out[1][f]), f
        assert math.isfinite(float(np.max(out[1][f])))
