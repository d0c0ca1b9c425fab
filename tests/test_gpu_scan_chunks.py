"""The FP64 line sweeps of the 3D solver in one pass over chunks with lead-in lines: the predictor's
velocity on the GPU against the oracle where the chunks can go wrong, a last chunk of one line,
lead-ins up to line 1 (large time step, small Re: weak diagonal dominance) and of a few lines, rows
of one to eight per lane of either direction with the last lane in use part full, chunks of 8 and of
16 lines.  Tolerance: 1e-12, that of the predictor's stages.  A value that is not finite is reported
by the entry point that runs the sweeps alone, and a later call with good fields is not affected."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(ni, nj, nk, re, dt):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    (xg, yg, zg), ic = make_case(ni, nj, nk, h1=0.01, r_out=10.0, sigma=0.05, seed=41)
    s = Solver3D(ni, nj, nk, re, dt, xg, yg, zg)
    state = [ic[k] for k in ("u", "v", "w", "p", "nlx", "nly", "nlz")]
    s.set_state(*state)
    return s, state, (xg, yg, zg)


def _predict(s):
    s.begin_step()
    for f in (s.contra_vel, s.nl, s.stress_tensor_dy, s.dif, s.p_source, s.iter_u):
        f()


@pytest.mark.parametrize("ni,nj,nk,re,dt", [(18, 35, 6, 100.0, 0.02), (34, 97, 5, 3900.0, 1e-3),
                                            (130, 82, 5, 100.0, 0.02), (42, 258, 5, 200.0, 0.01),
                                            (74, 121, 49, 100.0, 0.02), (323, 35, 5, 100.0, 0.02),
                                            (26, 449, 5, 200.0, 0.01), (450, 33, 5, 3900.0, 1e-3)])
def test_one_pass_sweeps(ni, nj, nk, re, dt):
    from oracle.oracle3d import Oracle3D
    s, state, nodes = _solver(ni, nj, nk, re, dt)
    _predict(s)
    o = Oracle3D(ni, nj, nk, re, dt, math.pi, *nodes)
    o.set_state(*state)
    for f in (o.pred_nl, o.pred_sgs, o.pred_dif_ps, o.pred_iter_u):
        f()
    inner = (slice(1, ni), slice(1, nj), slice(1, nk))
    for c in "uvw":
        a, b = s.get(c)[inner], o.array(c)[inner]
        err = np.abs(a - b).max() / np.abs(b).max()
        assert err < 1e-12, (c, err)


def test_value_that_is_not_finite():
    from fvm_amd import capi
    s, state, _ = _solver(34, 49, 9, 3900.0, 1e-3)
    _predict(s)
    good = s.get("u")
    bad = good.copy()
    bad[7, 9, 4] = np.nan
    s.set("difx", bad)
    with pytest.raises(capi.FvmError) as e:
        s.iter_u()
    assert e.value.code == 3
    s.set_state(*state)
    _predict(s)
    assert np.array_equal(s.get("u"), good)
