"""The transposed AF sweeps by chunks of eight lines, each with the lines before it that still count:
the adjoint gradient against central differences of the objective where the chunks can go wrong, a
last chunk of one line, fewer lines than a chunk's lead-in, rows of one to two per lane, and a large
time step and small Re (weak diagonal dominance: lead-ins of most of the plane) next to a small one
(lead-ins of a few lines).  Tolerance: that of the short-horizon gradient, 1e-5 of the largest
component (central differences with h = 1e-6 of sums rounded to 1e-16)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = 1e-6


@pytest.mark.parametrize("ni,nj,re,dt", [(10, 25, 40.0, 0.02), (18, 73, 40.0, 0.02),
                                         (66, 121, 60.0, 0.01), (34, 97, 400.0, 5e-4)])
def test_gradient_with_chunked_sweeps(ni, nj, re, dt):
    from fvm_amd.adjoint import DragProblem
    from fvm_amd.batch2d import Batch2D
    from fvm_amd.grid import make_case
    (xg, yg, _), ic = make_case(ni, nj, 1, h1=0.01, r_out=10.0, sigma=1e-3, seed=3)
    b = Batch2D([dict(ni=ni, nj=nj, re=re, dt=dt, xg=xg[:, :, 0], yg=yg[:, :, 0])],
                resimax=1e-14, npass=6)
    x0 = [tuple(ic[k][:, :, 0] for k in ("u", "v", "p", "nlx", "nly"))]
    pr = DragProblem(b, x0, 6, 3, tol=1e-13, maxpass=60)
    c = np.random.default_rng(5).normal(0.0, 0.01, (1, 128))
    pr.run(c)
    g = pr.gradient(c)[0]
    assert np.isfinite(g).all() and np.abs(g).max() > 0.0
    for k in np.random.default_rng(1).choice(128, 6, replace=False):
        e = np.zeros_like(c)
        e[0, k] = H
        fd = (pr.run(c + e, keep=False)[0] - pr.run(c - e, keep=False)[0]) / (2 * H)
        assert abs(g[k] - fd) <= 1e-5 * np.abs(g).max(), (k, g[k], fd)
