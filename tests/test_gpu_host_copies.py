"""Field copies through the pinned slots: values come back as they were set, for field sizes below,
at and above the slot size (2 MiB) and the ring's chunk changes (8 MiB), when the host array is
reused at once, when an upload is followed by a download, and in a batch of uneven sizes; the
history of a batch over the ring's end.  Equality is exact: nothing is computed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# cells with ghosts x 8 B: 1 kB, just below / above 2 MiB, several MiB, above 8 MiB
@pytest.mark.parametrize("ni,nj,nk", [(4, 4, 3), (63, 63, 63), (63, 64, 63), (90, 81, 65),
                                      (129, 129, 65)])
def test_fields_round_trip(ni, nj, nk):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    (xg, yg, zg), _ = make_case(ni, nj, nk, h1=0.01, r_out=10.0, sigma=0.0)
    s = Solver3D(ni, nj, nk, 3900.0, 1e-3, xg, yg, zg)
    rng = np.random.default_rng(3)
    names = ("u", "v", "w", "p", "nlx")
    keep = {}
    a = np.empty(s.shape, order="F")
    for q in names:
        a[...] = rng.normal(size=s.shape)
        keep[q] = a.copy(order="F")
        s.set(q, a)
        a[...] = -1.0  # the caller's array is free when the call returns
    for q in names:
        assert np.array_equal(s.get(q), keep[q]), q
    s.set("u", keep["p"])
    assert np.array_equal(s.get("u"), keep["p"])


def test_batch_fields_and_history():
    from fvm_amd.batch2d import batch_from_cases
    from fvm_amd.grid import ensemble_cases
    cases = ensemble_cases(5)
    b = batch_from_cases(cases, dt_scale=0.1)
    for q, c in enumerate(cases):
        for f in ("u", "v", "p", "nlx", "nly"):
            assert np.array_equal(b.get(q, f), c["ic"][f][:, :, 0]), (q, f)
    b.step(3)
    h = b.history(3)
    one = b.step(1)
    h4 = b.history(4)
    assert np.array_equal(h4[:3], h)
    assert [i["cd"] for i in one] == list(h4[3, :, 0])
    b.step(4096)
    tail = b.step(2)
    h = b.history(4096)
    assert [i["cd"] for i in tail] == list(h[-1, :, 0])
    assert np.array_equal(b.history(2), h[-2:])
