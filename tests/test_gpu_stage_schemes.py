"""pxt16's methods and K2 diffusion in one launch per RK stage
(csrc/imx_stage.hip): meshes below, at and past one block, the forms of each
scheme, each block size, against the FP64_REF handle; and the combinations
that keep the passes."""
import pytest

from imodel_amd.swm import Mesh, Swm
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

# the fused paths' tolerances with scheme options: tendency, h and u after 6 steps
TOL = {"fp64": (1e-12, 1e-12, 1e-11), "fp32": (5e-5, 1e-6, 1e-5)}


def evaluate(m, prec, dt, kw, kernels=None, sfc=True, tune=False, topo=False, coriolis=(0, 0.0)):
    h, u = m.spectral(34)
    with Swm(m, precision=prec, dt=dt, use_sfc=sfc) as s:
        s.set_scheme(**kw)
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


SCHEMES = {"pxt16": {"wrap": "pxt16"}, "k2": {"k2": 1e5, "diffus": "const"}}


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("glevel", [0, 1, 2, 4, 6])
@pytest.mark.parametrize("scheme", list(SCHEMES))
def test_sizes(scheme, glevel, prec):
    """As for the plain scheme, the three passes on the mesh's own numbering
    are the reference at glevel 6."""
    print("[gpu-case] stage", scheme, glevel, prec, flush=True)
    m = Mesh.icos(glevel)
    dt = min(300.0, 14400.0 / 2 ** glevel)
    kw = SCHEMES[scheme]
    ref = evaluate(m, "fp64_ref", dt, kw) if glevel < 6 else evaluate(m, prec, dt, kw, sfc=False, kernels=3)
    compare(evaluate(m, prec, dt, kw, kernels=1), ref, prec)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("kw,opt,kernels", [
    ({"wrap": "pxt16"}, {"topo": True, "tune": True}, 1),
    ({"wrap": "pxt16"}, {"coriolis": (1, 1e-4)}, 1),
    ({"wrap": "pxt16", "stag": "HC"}, {}, 3),
    ({"wrap": "pxt16", "pv": "apvm", "pvspar": 0.5}, {}, 3),
    ({"k2": 1e6, "diffus": "align"}, {"topo": True, "tune": True}, 1),
    ({"k2": 1e6, "diffus": "diam", "stag": "HC"}, {}, 1),
    ({"k2": 1e6, "diffus": "const"}, {"coriolis": (2, 1e-4)}, 1),
    ({"k2": 1e5, "diffus": "const", "k4": 1e14, "hyperdiffus": "align"}, {}, 3),
], ids=str)
def test_options(kw, opt, kernels, prec):
    print("[gpu-case] stage options", kw, opt, prec, flush=True)
    m = Mesh.icos(4)
    compare(evaluate(m, prec, 300.0, kw, kernels=kernels, **opt),
            evaluate(m, "fp64_ref", 300.0, kw, **{k: v for k, v in opt.items() if k != "tune"}), prec)
