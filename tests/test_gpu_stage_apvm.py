"""APVM in one launch per RK stage (csrc/imx_stage.hip), whose blocks hold one
ring of cells and triangles more: meshes below, at and past one block, both
staggerings, each block size, against the FP64_REF handle; and the handle that
changes between the schemes with and without it."""
import numpy as np
import pytest

from imodel_amd.swm import Mesh, Swm
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

# the fused paths' tolerances with scheme options: tendency, h and u after 6 steps
TOL = {"fp64": (1e-12, 1e-12, 1e-11), "fp32": (5e-5, 1e-6, 1e-5)}


def evaluate(m, prec, dt, kernels=None, sfc=True, tune=False, topo=False, coriolis=(0, 0.0), **kw):
    h, u = m.spectral(33)
    with Swm(m, precision=prec, dt=dt, use_sfc=sfc) as s:
        s.set_scheme(pv="apvm", pvspar=0.5, **kw)
        s.set_coriolis(*coriolis)
        if topo:
            s.set_topography(200.0 * (1.0 + m.arrays["v_p"].reshape(-1, 3)[:, 0]))
        if tune:
            s.set_state(h, u)
            s.tune(1)
        mt, ft = s.tendency(h, u)
        s.set_state(h, u)
        s.step(6)
        hs, us = s.get_state()
        if kernels:
            assert len(s.profile(1)) == kernels
        return mt, ft, hs, us


def compare(got, ref, prec):
    t, th, tu = TOL[prec]
    for g, r, tol in zip(got, ref, (t, t, th, tu)):
        assert rel_l2(g, r) < tol, rel_l2(g, r)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("glevel", [0, 1, 2, 3, 4, 6])
def test_sizes(glevel, prec):
    """As for the plain scheme, the three passes on the mesh's own numbering
    are the reference at glevel 6."""
    print("[gpu-case] stage apvm", glevel, prec, flush=True)
    m = Mesh.icos(glevel)
    dt = min(300.0, 14400.0 / 2 ** glevel)
    ref = evaluate(m, "fp64_ref", dt) if glevel < 6 else evaluate(m, prec, dt, sfc=False, kernels=3)
    compare(evaluate(m, prec, dt, kernels=1), ref, prec)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("kw", [{"stag": "HC"}, {"stag": "HC", "coriolis": (1, 1e-4)}, {"topo": True},
                                {"tune": True}], ids=lambda kw: "-".join(kw))
def test_options(kw, prec):
    print("[gpu-case] stage apvm options", kw, prec, flush=True)
    m = Mesh.icos(4)
    compare(evaluate(m, prec, 300.0, kernels=1, **kw),
            evaluate(m, "fp64_ref", 300.0, **{k: v for k, v in kw.items() if k != "tune"}), prec)


def test_schemes_in_turn():
    """APVM, the plain scheme, APVM with diffusion (three passes), another
    staggering and APVM again: the first tendency bit for bit."""
    print("[gpu-case] stage apvm in turn", flush=True)
    m = Mesh.icos(4)
    h, u = m.spectral(5)
    with Swm(m, precision="fp32", dt=600.0) as s:
        plain = s.tendency(h, u)
        s.set_scheme(pv="apvm", pvspar=0.5)
        first = s.tendency(h, u)
        assert not np.array_equal(first[1], plain[1])
        for kw in ({}, {"pv": "apvm", "k2": 1e5}, {"stag": "HC", "pv": "apvm"}, {"wrap": "pxt16"}):
            s.set_scheme(**kw)
            s.tendency(h, u)
        s.set_scheme(pv="apvm", pvspar=0.5)
        again = s.tendency(h, u)
        s.set_scheme()
        back = s.tendency(h, u)
    assert all(np.array_equal(a, b) for a, b in zip(first, again))
    assert all(np.array_equal(a, b) for a, b in zip(plain, back))
