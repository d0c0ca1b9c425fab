"""A change of the time step forms the lead-in tables of the one-pass FP64 line sweeps anew: steps after
it equal, bit for bit, those of a solver made with that time step, from strong to weak diagonal
dominance (lead-ins of a few lines, and of most of the plane) and back, in 3D with the temperature's
lines and in the batched 2D solver."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _box(dt, then=None):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    ni, nj, nk = 34, 73, 5
    (xg, yg, zg), ic = make_case(ni, nj, nk, h1=0.01, r_out=10.0, sigma=0.01, seed=41)
    s = Solver3D(ni, nj, nk, 60.0, dt, xg, yg, zg, poisson_mode=2, nswpp=50, resimax=1e-8)
    t = np.asfortranarray(0.5 + 0.1 * ic["u"])
    s.set_temperature(t, np.zeros_like(t), 40.0)
    if then:
        s.set_dtime(then)
    s.set_state(*[ic[k] for k in ("u", "v", "w", "p", "nlx", "nly", "nlz")])
    for _ in range(2):
        s.step()
    return [s.get(q) for q in "uvwpt"]


def _plane(dt, then=None):
    from fvm_amd.batch2d import Batch2D
    from fvm_amd.grid import make_case
    (xg, yg, _), ic = make_case(42, 97, 1, h1=0.01, r_out=10.0, sigma=1e-3, seed=3)
    b = Batch2D([dict(ni=42, nj=97, re=40.0, dt=dt, xg=xg[:, :, 0], yg=yg[:, :, 0])], mixed=False)
    if then:
        b.set_dtime(0, then)
    b.set_state(0, *[ic[k][:, :, 0] for k in ("u", "v", "p", "nlx", "nly")])
    b.step(3)
    return [b.get(0, q) for q in "uvp"]


@pytest.mark.parametrize("run", [_box, _plane])
@pytest.mark.parametrize("a,b", [(1e-4, 0.01), (0.01, 1e-4)])
def test_leads_follow_the_time_step(run, a, b):
    for x, y in zip(run(a, b), run(b)):
        assert np.isfinite(x).all() and np.array_equal(x, y)
