"""A case of the FP64 batched 2D solver gives the same bits alone and in a batch of many, on either side of
the number of wavefronts that fill the chip: the lines at which its sweeps start are its own.  Fields of
1e-27 to 1 side by side, where what a lead-in leaves out (1e-20 of the largest value) can reach a last
bit, at strong to weak diagonal dominance.  No tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cases():
    from fvm_amd.grid import make_case
    specs, x0 = [], []
    for q in range(112, 128):
        gen = np.random.default_rng(100 + q)
        ni, nj = [(97, 385), (34, 257), (18, 129), (193, 65)][q % 4]
        dt, re = 10.0 ** gen.uniform(-6, -2.5), 10.0 ** gen.uniform(0.7, 2.3)
        h1 = [0.03, 0.01][q // 4 % 2]
        (xg, yg, _), ic = make_case(ni, nj, 1, h1=h1, r_out=20.0, sigma=1e-3, seed=11 + q)
        specs.append(dict(ni=ni, nj=nj, re=re, dt=dt, xg=xg[:, :, 0], yg=yg[:, :, 0]))
        x = [ic[k][:, :, 0] for k in ("u", "v", "p", "nlx", "nly")]
        w = gen.uniform(6, 30)
        for m in (0, 1):
            x[m] = np.asfortranarray(gen.normal(size=(ni + 1, nj + 1))
                                     * 10.0 ** -gen.uniform(0.0, w, (ni + 1, nj + 1)))
        if q // 8 % 2:
            x[2:] = [np.zeros_like(a) for a in x[2:]]
        x0.append(x)
    return specs, x0


def _run(specs, x0):
    from fvm_amd.batch2d import Batch2D
    b = Batch2D(specs, mixed=False, resimax=1e-8)
    for c, x in enumerate(x0):
        b.set_state(c, *x)
    b.step(1)
    return [[b.get(c, f) for f in "uvp"] for c in range(b.n)]


def test_alone_and_among_many():
    specs, x0 = _cases()
    many = _run(specs * 4, x0 * 4)
    for q in range(len(specs)):
        one = _run(specs[q:q + 1], x0[q:q + 1])[0]
        for f, a, b in zip("uvp", one, many[q]):
            assert np.isfinite(a).all() and np.array_equal(a, b), (q, f, int((a != b).sum()))
