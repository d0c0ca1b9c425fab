"""Field copies of one context from several threads at once (a program that writes a dump on one thread
and reads probes on another): every thread gets the values of the field it asked for, and what each
sets arrives, for fields that take one pinned slot and for fields that take the ring; and copies
through a ring whose slots are used several times over.  Equality is exact: nothing is computed."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(ni, nj, nk):
    from fvm_amd.grid import make_case
    from fvm_amd.solver import Solver3D
    (xg, yg, zg), _ = make_case(ni, nj, nk, h1=0.01, r_out=10.0, sigma=0.0)
    return Solver3D(ni, nj, nk, 3900.0, 1e-3, xg, yg, zg)


# 35 kB, 0.5 MB, 3.2 MB
@pytest.mark.parametrize("ni,nj,nk", [(12, 17, 18), (34, 49, 33), (66, 129, 45)])
def test_threads_share_a_context(ni, nj, nk):
    s = _solver(ni, nj, nk)
    names = ("u", "v", "w", "p")
    val = {q: np.asfortranarray(np.random.default_rng(k).normal(size=s.shape))
           for k, q in enumerate(names)}
    wrong = []

    def work(q):
        for _ in range(12):
            s.set(q, val[q])
            if not np.array_equal(s.get(q), val[q]):
                wrong.append(q)

    pool = [threading.Thread(target=work, args=(q,)) for q in names]
    for t in pool:
        t.start()
    for t in pool:
        t.join()
    assert not wrong


# 5.3 MB: eleven chunks of 512 KiB; 17.4 MB: nine of 2 MiB (eight slots each)
@pytest.mark.parametrize("ni,nj,nk", [(129, 129, 38), (129, 129, 127)])
def test_ring_slots_used_again(ni, nj, nk):
    s = _solver(ni, nj, nk)
    rng = np.random.default_rng(9)
    a = np.asfortranarray(rng.normal(size=s.shape))
    b = np.asfortranarray(rng.normal(size=s.shape))
    for _ in range(3):
        s.set("u", a)
        s.set("v", b)
        assert np.array_equal(s.get("u"), a) and np.array_equal(s.get("v"), b)
