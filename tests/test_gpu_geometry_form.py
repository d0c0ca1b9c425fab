"""The form of the geometry that a context's kernels work with: formed anew from one plane on extruded grids
from 2^19 cells, whatever the span's spacing (set-up compares it with the stored arrays bit for bit and
falls back to them where one bit of one cell differs), until the caller sets the volume or a metric;
stored arrays on smaller grids and on grids that are not extruded.  And steps of one grid in two forms
give equal fields."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PLANE, XZ0, STORED = "plane", "stored, xi_z = eta_z = 0", "stored"


def _z(span, nk):
    t = np.arange(nk) / (nk - 1)
    return {"pi": math.pi * t, "dyadic": 2.0 * t, "stretched": math.pi * t ** 1.3}[span]


def _solver(ni, nj, nk, span="pi", wave=0.0, **kw):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    (xg, yg, zg), ic = make_case(ni, nj, nk, h1=0.01, r_out=10.0, sigma=0.05, seed=7)
    zg = np.asfortranarray(np.broadcast_to(_z(span, nk)[None, None, :], xg.shape))
    f = 1.0 + wave * np.cos(2.0 * zg)
    s = Solver3D(ni, nj, nk, 3900.0, 1e-3, np.asfortranarray(xg * f), np.asfortranarray(yg * f), zg,
                 **kw)
    s.set_state(*[ic[k] for k in ("u", "v", "w", "p", "nlx", "nly", "nlz")])
    return s


@pytest.mark.parametrize("ni,nj,nk,span", [
    (12, 385, 129, "pi"), (66, 131, 65, "dyadic"), (66, 257, 33, "stretched"), (130, 67, 65, "pi"),
    (162, 129, 33, "pi"), (193, 257, 65, "pi"), (150, 209, 41, "pi")])
def test_large_extruded_grids(ni, nj, nk, span):
    s = _solver(ni, nj, nk, span)
    assert s.geometry_form == PLANE
    s.set("u", s.get("u"))
    s.set_dtime(5e-4)
    assert s.geometry_form == PLANE
    s.set("djac", s.get("djac"))
    assert s.geometry_form == XZ0


@pytest.mark.parametrize("name", ["xix", "etx", "ztx", "xiy", "ety", "zty", "xiz", "etz", "ztz"])
def test_a_metric_that_is_set_ends_the_form(name):
    s = _solver(66, 131, 65, "dyadic")
    assert s.geometry_form == PLANE
    s.set(name, s.get(name))
    assert s.geometry_form == STORED


def test_other_grids():
    assert _solver(97, 129, 17).geometry_form == XZ0
    assert _solver(66, 129, 59).geometry_form == XZ0  # 67 x 130 x 60 cells with ghosts: just below
    assert _solver(66, 131, 65, wave=0.05).geometry_form == STORED


@pytest.mark.parametrize("kw", [dict(poisson_mode=2, nswpp=50, resimax=1e-8),
                                dict(poisson_mode=3, af_mode=2, nswpp=50, resimax=1e-8)])
def test_equal_steps(kw):
    out = []
    for stored in (False, True):
        s = _solver(66, 131, 65, "dyadic", **kw)
        if stored:
            s.set("djac", s.get("djac"))
        assert s.geometry_form == (XZ0 if stored else PLANE)
        for _ in range(2):
            s.step()
        out.append([s.get(q) for q in "uvwp"])
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)
