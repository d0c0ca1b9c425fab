"""The one-pass FP64 line sweeps of the 3D solver in chunks of 32 lines, which grids with more than 65536
lines of u, v, w take (192 to 256 cells in two directions): the predictor's velocity on the GPU against
the oracle on thin grids of that many lines, I lines and J lines, with a last chunk of one line,
lead-ins of a few lines and (large time step, small Re) of many.  Tolerance: 1e-12, that of the
predictor's stages."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,re,dt", [(12, 354, 3900.0, 1e-3), (12, 354, 100.0, 0.02),
                                         (354, 17, 100.0, 0.02)])
def test_chunks_of_32_lines(ni, nj, re, dt):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    from oracle.oracle3d import Oracle3D
    nk = 65
    assert 3 * (nk - 1) * (max(ni, nj) - 1) > 65536 and (max(ni, nj) - 1) % 32 == 1
    (xg, yg, zg), ic = make_case(ni, nj, nk, h1=0.01, r_out=10.0, sigma=0.05, seed=41)
    state = [ic[k] for k in ("u", "v", "w", "p", "nlx", "nly", "nlz")]
    s = Solver3D(ni, nj, nk, re, dt, xg, yg, zg)
    s.set_state(*state)
    s.begin_step()
    for f in (s.contra_vel, s.nl, s.stress_tensor_dy, s.dif, s.p_source, s.iter_u):
        f()
    o = Oracle3D(ni, nj, nk, re, dt, math.pi, xg, yg, zg)
    o.set_state(*state)
    for f in (o.pred_nl, o.pred_sgs, o.pred_dif_ps, o.pred_iter_u):
        f()
    inner = (slice(1, ni), slice(1, nj), slice(1, nk))
    for c in "uvw":
        a, b = s.get(c)[inner], o.array(c)[inner]
        err = np.abs(a - b).max() / np.abs(b).max()
        assert err < 1e-12, (c, err)
