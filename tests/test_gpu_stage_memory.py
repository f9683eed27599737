"""The tables of the one-launch stage are on top of the passes': where they find
no memory (here: more than the handle allows them) every call that makes them
succeeds and the passes run."""
import numpy as np
import pytest

from imodel_amd.swm import Mesh, Swm
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

# the fused paths' tolerances with scheme options: tendency, h and u after 6 steps
TOL = {"fp64": (1e-12, 1e-12, 1e-11), "fp32": (5e-5, 1e-6, 1e-5)}
SCHEMES = [{}, {"pv": "apvm", "pvspar": 0.5}, {"stag": "HC"}, {"wrap": "gass18"}, {"wrap": "pxt16"},
           {"k2": 1e5, "diffus": "const"}, {}]


def evaluate(s, h, u):
    t = s.tendency(h, u)
    s.set_state(h, u)
    s.step(6)
    return t + s.get_state(), len(s.profile(1))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_no_memory_for_the_tables(prec):
    print("[gpu-case] stage tables without memory", prec, flush=True)
    m = Mesh.icos(4)
    h, u = m.spectral(36)
    with Swm(m, precision=prec, dt=300.0) as a, Swm(m, precision=prec, dt=300.0) as b:
        a.set_stage_limit(4096)
        for k, kw in enumerate(SCHEMES):
            for s in (a, b):
                s.set_scheme(**kw)
                s.set_coriolis(2 if k % 2 else 0, 1e-4)
            if k == 3:
                a.tune(1)
            (got, na), (want, nb) = evaluate(a, h, u), evaluate(b, h, u)
            assert na == 3 and nb == (3 if kw.get("wrap") == "gass18" else 1), kw
            t, th, tu = TOL[prec]
            for g, r, tol in zip(got, want, (t, t, th, tu)):
                assert rel_l2(g, r) < tol, (kw, rel_l2(g, r))
        a.set_stage_limit(0)
        (got, na), (want, _) = evaluate(a, h, u), evaluate(b, h, u)
        assert na == 1 and all(np.array_equal(g, r) for g, r in zip(got, want))


def test_tables_go_with_their_scheme():
    print("[gpu-case] stage tables given back", flush=True)
    m = Mesh.icos(4)
    with Swm(m, precision="fp32") as s:
        held = []
        for kw in ({"wrap": "gass18"}, {}, {"wrap": "gass18"}, {}):
            s.set_scheme(**kw)
            held.append(int(s.info()[3]))
    assert held[0] == held[2] and held[1] == held[3] > held[0] + 100 * m.nv
