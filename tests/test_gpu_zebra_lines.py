"""The FP64 zebra line sweeps: tests of the residual enqueued ahead of the one waited for, and the line
solves by factor scans at one to eight rows per lane with remainders.
* Sweeps ended by the tolerance leave the pressure, residual and count of sweeps ended by the cap at
  that count, to the last bit (those enqueued past the end change nothing), for every sweep tested
  and every third.
* The oracle's residual of the GPU's pressure is the one reported, to 1e-6 of it (the source comes
  from velocities that agree to 1e-12 of fields 1e3 to 1e5 times their residual's scale)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,nk,every", [(34, 25, 9, 1), (66, 41, 12, 3), (131, 33, 6, 1),
                                            (262, 33, 5, 3), (450, 17, 5, 1)])
def test_zebra_sweeps(ni, nj, nk, every):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    from oracle.oracle3d import Oracle3D
    (xg, yg, zg), ic = make_case(ni, nj, nk, h1=0.01, r_out=10.0, sigma=0.05, seed=23)
    state = [ic[k] for k in ("u", "v", "w", "p", "nlx", "nly", "nlz")]

    def sweeps(cap, tol):
        s = Solver3D(ni, nj, nk, 3900.0, 1e-3, xg, yg, zg, nswpp=cap, resimax=tol,
                     check_every=every)
        s.set_state(*state)
        s.begin_step()
        for f in (s.contra_vel, s.nl, s.stress_tensor_dy, s.dif, s.p_source, s.iter_u):
            f()
        s.correct(-1.0)
        s.contra_vel()
        r, n = s.iter_p()
        return r, n, s.get("p")

    r9, n9, _ = sweeps(9, 1e-30)
    assert n9 == 9 and 0.0 < r9 < 1.0
    r, n, p = sweeps(60, r9 * (1.0 + 1e-9))
    assert r <= r9 * (1.0 + 1e-9) and n <= 9 and n % every == 0, (r, n)
    rc, nc, pc = sweeps(n, 1e-30)
    assert (rc, nc) == (r, n) and np.array_equal(p, pc)
    o = Oracle3D(ni, nj, nk, 3900.0, 1e-3, math.pi, xg, yg, zg)
    o.set_state(*state)
    o.predictor(True)
    o.correct_predictor()
    o.array("p")[:, :, :] = p
    assert abs(o.p_residual() - r) <= 1e-6 * r
