"""State slots of the batched 2D solver (one copy launch over every plane: odd and even plane sizes,
several cases) give the planes back bit for bit, and the adjoint step's Poisson solve stops by the
device's flag as by the host's test: with one case and with several, before the first correction,
after one, and at the pass limit.  No tolerance: a case's result does not depend on the others, and
two equal cases take the passes of one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(cases):
    from fvm_amd.batch2d import Batch2D
    from fvm_amd.grid import make_case
    specs, x0 = [], []
    for ni, nj, re, seed in cases:
        (xg, yg, _), ic = make_case(ni, nj, 1, h1=0.01, r_out=10.0, sigma=1e-3, seed=seed)
        specs.append(dict(ni=ni, nj=nj, re=re, dt=0.002, xg=xg[:, :, 0], yg=yg[:, :, 0]))
        x0.append(tuple(ic[k][:, :, 0] for k in ("u", "v", "p", "nlx", "nly")))
    b = Batch2D(specs, resimax=1e-12, npass=6)
    for c, x in enumerate(x0):
        b.set_state(c, *x)
    return b


def _state(b):
    return [b.get(c, k) for c in range(b.n) for k in ("u", "v", "p", "nlx", "nly")]


def test_slots_give_the_state_back():
    b = _batch([(10, 25, 40.0, 1), (18, 73, 80.0, 2), (65, 97, 100.0, 3)])
    start = _state(b)
    b.save(0)
    b.step(3)
    later = _state(b)
    b.save(3)
    b.load(0)
    assert all(np.array_equal(p, q) for p, q in zip(_state(b), start))
    b.load(3)
    assert all(np.array_equal(p, q) for p, q in zip(_state(b), later))
    assert not all(np.array_equal(p, q) for p, q in zip(start, later))


@pytest.mark.parametrize("tol,maxpass", [(1.0, 50), (1e-13, 50), (1e-6, 1), (1e-30, 3)])
def test_adjoint_poisson_stops_alike_for_one_case_and_two(tol, maxpass):
    out = []
    for n in (1, 2):
        b = _batch([(18, 73, 80.0, 2)] * n)
        b.adjoint_init()
        b.step(2)
        r = [b.adjoint_step(np.zeros(n), tol, maxpass)]
        assert r[0] == 0.0  # a zero objective leaves the zero state
        assert all(not b.adjoint_state(0, k).any() for k in ("u", "v", "p"))
        r += [b.adjoint_step(np.ones(n), tol, maxpass) for _ in range(2)]
        out.append((r, [b.adjoint_state(n - 1, k) for k in ("u", "v", "p", "nlx", "nly")]))
    assert out[0][0] == out[1][0]
    assert all(np.array_equal(p, q) for p, q in zip(out[0][1], out[1][1]))
    assert out[0][1][0].any()
    if tol == 1.0:
        assert out[0][0][1] == 1.0  # mu = 0: no correction
    elif maxpass > 1 and tol > 1e-20:
        assert max(out[0][0]) <= tol
