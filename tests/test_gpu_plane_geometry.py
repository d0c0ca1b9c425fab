"""Steps whose kernels form the metrics of an extruded grid anew from its cross-section against the
same steps with the stored arrays (which a context uses once its volume field has been set, here to
what it was).  Both must agree to the last bit: the set-up checks that the metrics formed anew equal
the stored ones, and the terms left out are products with exact zeros.  Spans: pi (the rounding of z
gives planes of several different metrics), a power of two over a power of two (a single one),
stretched (all different).  Sizes, all of them with the half million cells from which the form is
used: few columns next to the I boundaries, an I tile of one cell, J remainders, a K line of 64."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _z(span, nk):
    t = np.arange(nk) / (nk - 1)
    return {"pi": math.pi * t, "dyadic": 2.0 * t, "stretched": math.pi * t ** 1.3}[span]


@pytest.mark.parametrize("ni,nj,nk,span,form,thermal", [
    (12, 385, 129, "pi", "zebra", False),
    (66, 131, 65, "dyadic", "fp64", False),
    (66, 257, 33, "stretched", "zebra", True),
    (130, 67, 65, "pi", "mixed", False),
    (162, 129, 33, "pi", "fp64", True),
])
def test_plane_form_equals_stored_geometry(ni, nj, nk, span, form, thermal):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    (xg, yg, zg), ic = make_case(ni, nj, nk, h1=0.01, r_out=10.0, sigma=0.05, seed=7)
    zg = np.asfortranarray(np.broadcast_to(_z(span, nk)[None, None, :], xg.shape))
    kw = dict(mixed=dict(poisson_mode=3, af_mode=2), fp64=dict(poisson_mode=2),
              zebra=dict(af_mode=2))[form]
    t = np.asfortranarray(0.5 + 0.1 * ic["u"])
    out = []
    for stored in (False, True):
        s = Solver3D(ni, nj, nk, 3900.0, 1e-3, xg, yg, zg, nswpp=20, resimax=1e-8, **kw)
        s.set_state(*[ic[k] for k in ("u", "v", "w", "p", "nlx", "nly", "nlz")])
        if thermal:
            s.set_temperature(t, np.zeros_like(t))
        if stored:
            s.set("djac", s.get("djac"))
        for _ in range(3):
            s.step()
        names = ["u", "v", "w", "p", "nlx", "dify", "s_u", "s_w"] + (["t"] if thermal else [])
        out.append([s.get(q) for q in names])
    for q, a, b in zip(names, *out):
        assert np.isfinite(a).all() and np.array_equal(a, b), (q, np.abs(a - b).max())
