"""States moved by several threads at once: the instances of an ensemble, and
the readers and tendency calls of one handle, share a staging area."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from imodel_amd.swm import H0_GEO, Ensemble, Mesh, Swm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_instances_from_threads(prec):
    print("[gpu-case] ensemble states from threads", prec, flush=True)
    meshes = {g: Mesh.icos(g) for g in (2, 4, 6)}
    ms = [meshes[(2, 4, 6)[i % 3]] for i in range(12)]  # the area grows under way
    x = [m.spectral(100 + i) for i, m in enumerate(ms)]
    with Ensemble(ms, [100.0] * len(ms), precision=prec, h_ref=H0_GEO) as E, ThreadPoolExecutor(8) as pool:
        one = []
        for i, (h, u) in enumerate(x):
            E.set_state(i, h, u)
            one.append(E.get_state(i))
        zero = [np.zeros_like(a) for m in ms for a in (np.zeros(m.nv), np.zeros(m.ne))]
        for _ in range(4):
            list(pool.map(lambda i: E.set_state(i, zero[2 * i], zero[2 * i + 1]), range(len(ms))))
            list(pool.map(lambda i: E.set_state(i, *x[i]), range(len(ms))))
            for got, want in zip(pool.map(E.get_state, range(len(ms))), one):
                assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("prec", ["fp64_ref", "fp64", "fp32"])
def test_one_handle_from_threads(prec):
    print("[gpu-case] one handle from threads", prec, flush=True)
    m = Mesh.icos(5)
    h, u = m.spectral(3)
    xs = [m.spectral(10 + k) for k in range(4)]
    with Swm(m, precision=prec, dt=300.0, h_ref=H0_GEO) as s, ThreadPoolExecutor(8) as pool:
        s.set_state(h, u)
        state, tend = s.get_state(), [s.tendency(*x) for x in xs]
        for _ in range(4):
            reads = [pool.submit(s.get_state) for _ in range(8)]
            calls = [pool.submit(s.tendency, *xs[k % 4]) for k in range(8)]
            for r in reads:
                assert all(np.array_equal(a, b) for a, b in zip(r.result(), state))
            for k, c in enumerate(calls):
                assert all(np.array_equal(a, b) for a, b in zip(c.result(), tend[k % 4]))
