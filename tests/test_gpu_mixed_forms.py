"""Runs whose FP64 part feeds an FP32 one keep the results of earlier versions: the FP32 part rounds a
residual of the FP64 fields, so operands that differ in their last bit come out 1e-12 to 1e-7 apart.
The fields of a few steps against those recorded on an MI355X with the version in which every form took
its lines by chunk passes, the pressure lines by reduction and the model's sums by 16 planes (python
tests/test_gpu_mixed_forms.py writes the records of the version at hand).  Equality is exact: runs of
one version repeat to the bit, and so must the same operations in the same order."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _slab(ni, nj, re, dt, steps, **kw):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver2D
    (xg, yg, _), ic = make_case(ni, nj, 1, h1=0.01, r_out=20.0, sigma=1e-3, seed=5)
    s = Solver2D(ni, nj, re, dt, xg[:, :, 0], yg[:, :, 0], nswpp=50, **kw)
    s.set_state(*[ic[k][:, :, 0] for k in ("u", "v", "p", "nlx", "nly")])
    for _ in range(steps):
        s.step()
    return {q: s.get(q) for q in "up"}


def _batch(cases, steps, **kw):
    from fvm_amd.batch2d import Batch2D
    from fvm_amd.grid import make_case
    specs, x0 = [], []
    for ni, nj, re, dt in cases:
        (xg, yg, _), ic = make_case(ni, nj, 1, h1=0.01, r_out=20.0, sigma=1e-3, seed=5)
        specs.append(dict(ni=ni, nj=nj, re=re, dt=dt, xg=xg[:, :, 0], yg=yg[:, :, 0]))
        x0.append([ic[k][:, :, 0] for k in ("u", "v", "p", "nlx", "nly")])
    b = Batch2D(specs, **kw)
    for c, x in enumerate(x0):
        b.set_state(c, *x)
    b.step(steps)
    return {f"{q}{c}": b.get(c, q) for c in range(b.n) for q in "up"}


def _les(ni, nj, nk, steps, use_les, **kw):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    (xg, yg, zg), ic = make_case(ni, nj, nk, h1=0.004, r_out=20.0, sigma=0.05, seed=7)
    s = Solver3D(ni, nj, nk, 3900.0, 1e-3, xg, yg, zg, use_les=use_les, nswpp=50, **kw)
    s.set_state(*[ic[k] for k in ("u", "v", "w", "p", "nlx", "nly", "nlz")])
    for _ in range(steps):
        s.step()
    return {q: s.get(q) for q in "up"}


# rows of a line per lane: one to five; last chunks of one line and of a whole one; weak dominance
FORMS = {
    # FP64 line sweeps, FP32 pressure corrections
    "slab_sep32": lambda: _slab(50, 65, 100.0, 1e-3, 12, poisson_mode=3, resimax=1e-8),
    "slab_sep32_long": lambda: _slab(18, 289, 200.0, 1e-3, 8, poisson_mode=3, resimax=1e-8),
    "slab_sep32_weak": lambda: _slab(82, 97, 40.0, 1e-2, 8, poisson_mode=3, resimax=1e-8),
    "slab_zebra32": lambda: _slab(34, 97, 100.0, 1e-3, 8, poisson_mode=1, resimax=1e-4),
    "batch_sep32": lambda: _batch([(50, 65, 100.0, 1e-3), (18, 289, 200.0, 1e-3),
                                   (82, 97, 40.0, 1e-2)], 8),
    "box_sep32": lambda: _les(35, 49, 5, 6, False, poisson_mode=3, resimax=1e-8),
    # FP32 line sweeps (change form), FP64 pressure by line relaxation
    "slab_af32_zebra": lambda: _slab(50, 65, 100.0, 1e-3, 12, poisson_mode=0, af_mode=2,
                                     resimax=1e-4),
    "box_af32_zebra": lambda: _les(26, 33, 5, 6, False, poisson_mode=0, af_mode=2, resimax=1e-4),
    # the model's sums, FP64 line sweeps (chunk passes, and the exact order), FP32 pressure corrections
    "les_sep32": lambda: _les(22, 49, 17, 12, True, poisson_mode=3, resimax=1e-8),
    "les_exact_sep32": lambda: _les(18, 33, 17, 8, True, poisson_mode=3, af_mode=1, resimax=1e-8),
}


def _path(form):
    return os.path.join(GOLDEN, f"mixed_{form}.npz")


@pytest.mark.parametrize("form", FORMS)
def test_fields_of_earlier_versions(form):
    got = FORMS[form]()
    with np.load(_path(form), allow_pickle=False) as z:
        assert sorted(z.files) == sorted(got)
        for k in z.files:
            e = np.linalg.norm(got[k] - z[k]) / np.linalg.norm(z[k])
            assert np.isfinite(got[k]).all() and np.array_equal(got[k], z[k]), (form, k, e)


if __name__ == "__main__":
    for name, run in FORMS.items():
        np.savez_compressed(_path(name), **run())
        print(name, flush=True)
