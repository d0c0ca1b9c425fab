"""Planes per workgroup of the K-marching stencil kernels chosen by the grid size: the predictor's
stages on the GPU against the oracle (C restatement of the reference's step) where the choice and
its remainders can go wrong: one plane per workgroup with partial tiles, a few planes with a
shorter last group (130 x 64 x 48 cells: 3 and 5 planes), an I tile of one cell, a two-plane
span.  Tolerances: the reference's association order is kept, 1e-14 for the convective, diffusive
and pressure terms; 1e-12 where the dynamic coefficient's sum is grouped differently."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,nk", [(12, 9, 3), (34, 31, 8), (66, 41, 20), (131, 65, 49)])
def test_predictor_stages(ni, nj, nk):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    from oracle.oracle3d import Oracle3D
    (xg, yg, zg), ic = make_case(ni, nj, nk, h1=0.01, r_out=10.0, sigma=0.05, seed=31)
    state = [ic[k] for k in ("u", "v", "w", "p", "nlx", "nly", "nlz")]
    s = Solver3D(ni, nj, nk, 3900.0, 1e-3, xg, yg, zg)
    s.set_state(*state)
    o = Oracle3D(ni, nj, nk, 3900.0, 1e-3, math.pi, xg, yg, zg)
    o.set_state(*state)
    inner = (slice(1, ni), slice(1, nj), slice(1, nk))

    def check(names, tol):
        for c in names:
            a, b = s.get(c)[inner], o.array(c)[inner]
            err = np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)
            assert err < tol, (ni, nj, nk, c, err)

    s.begin_step()
    s.contra_vel()
    s.nl()
    o.pred_nl()
    check(("nlx", "nly", "nlz"), 1e-14)
    c_avg = s.stress_tensor_dy()
    o.pred_sgs()
    assert abs(c_avg - o.scalar("c_avg")) <= 1e-12 * abs(o.scalar("c_avg"))
    check(("nut", "sgsx", "sgsy", "sgsz", "nlx", "nly", "nlz"), 1e-12)
    s.dif()
    s.p_source()
    o.pred_dif_ps()
    check(("difx", "dify", "difz", "s_u", "s_v", "s_w"), 1e-14)
    s.iter_u()
    o.pred_iter_u()
    check(("u", "v", "w"), 1e-12)
    s.correct(-1.0)
    o.correct_predictor()
    check(("u", "v", "w"), 1e-12)
