"""FP64 zebra sweeps: however seldom the residual is tested, at most three sweeps are enqueued past the
test that ends them, and the sweeps, residual and pressure are those of a test after every sweep.  No
tolerance: counts and bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _iter_p(every, cap, tol):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    ni, nj, nk = 34, 33, 9
    (xg, yg, zg), ic = make_case(ni, nj, nk, h1=0.01, r_out=10.0, sigma=0.05, seed=23)
    s = Solver3D(ni, nj, nk, 3900.0, 1e-3, xg, yg, zg, nswpp=cap, resimax=tol, check_every=every)
    s.set_state(*[ic[k] for k in ("u", "v", "w", "u", "nlx", "nly", "nlz")])  # a pressure not zero
    s.begin_step()
    for f in (s.contra_vel, s.nl, s.stress_tensor_dy, s.dif, s.p_source, s.iter_u):
        f()
    s.correct(-1.0)
    s.contra_vel()
    s.profile(True)
    s.profile_reset()
    r, n = s.iter_p()
    calls = s.profile_get().get("p_sweep64", (0.0, 0))[1]
    return r, n, calls, s.get("p")


@pytest.mark.parametrize("every", [1, 2, 3, 4, 7, 50])
def test_sweeps_past_the_end(every):
    r, n, calls, _ = _iter_p(every, 400, 1e300)  # the first test ends them
    assert n == 0 and calls <= 3, (n, calls)
    tol = 0.01 * r
    r, n, calls, p = _iter_p(every, 400, tol)
    assert r <= tol and 0 < n < 400 and n % every == 0 and calls <= n + 3, (r, n, calls)
    rc, nc, calls, pc = _iter_p(1, n, 0.0)  # the same sweeps, ended by the cap
    assert calls == n
    assert (rc, nc) == (r, n) and np.array_equal(p, pc)
