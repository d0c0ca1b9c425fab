"""The FP64 AF sweeps of the batched 2D solver by chunks with lead-in lines: one step against the CPU
oracle on the 2D slab where the chunks can go wrong, a last chunk of one line, lead-ins up to line 1
(large time step and small Re: weak diagonal dominance) and of a few lines, rows of one to seven per
lane with the last lane in use part full.  Tolerance: 1e-10 of the field maximum, that of the long
lines' step (the pressure converged to 1e-12)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LZ = 1.0e6


@pytest.mark.parametrize("ni,nj,re,dt", [(10, 25, 40.0, 0.02), (82, 97, 40.0, 0.01),
                                         (150, 73, 400.0, 5e-4), (34, 289, 100.0, 0.005),
                                         (66, 433, 180.0, 0.0025)])
def test_sweeps_against_oracle_slab(ni, nj, re, dt):
    from fvm_amd.batch2d import Batch2D
    from fvm_amd.grid import make_case
    from oracle.oracle3d import Oracle3D

    def slab(a, planes):
        return np.asfortranarray(np.repeat(np.asarray(a)[:, :, None], planes, axis=2))

    (xg, yg, _), ic = make_case(ni, nj, 1, h1=0.01, r_out=20.0, sigma=1e-3, seed=17)
    xg, yg = xg[:, :, 0], yg[:, :, 0]
    st = [ic[k][:, :, 0] for k in ("u", "v", "p", "nlx", "nly")]
    b = Batch2D([dict(ni=ni, nj=nj, re=re, dt=dt, xg=xg, yg=yg)], mixed=False, resimax=1e-12,
                npass=8)
    b.set_state(0, *st)
    info = b.step(1)[0]
    assert info["status"] == 0 and info["resip"] <= 1e-12, info
    zg = np.zeros((ni, nj, 2), order="F")
    zg[:, :, 1] = LZ
    o = Oracle3D(ni, nj, 2, re, dt, LZ, slab(xg, 2), slab(yg, 2), zg)
    o.set_no_pref(True)
    z = np.zeros((ni + 1, nj + 1, 3), order="F")
    o.set_state(slab(st[0], 3), slab(st[1], 3), z, slab(st[2], 3), slab(st[3], 3),
                slab(st[4], 3), z)
    o.predictor(False)
    o.correct_predictor()
    o.array("p")[:, :, :] = slab(b.get(0, "p"), 3)
    assert o.p_residual() <= 1e-10
    o.finish_step()
    for c in ("u", "v"):
        ref = o.array(c)[:, :, 1]
        err = np.abs(b.get(0, c) - ref).max() / np.abs(ref).max()
        assert err < 1e-10, (c, err)
