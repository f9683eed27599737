"""The pressure gradient of the one-launch stage (csrc/imx_stage.hip): from rest
the momentum tendency is the jump of the potential times 1 / (|e| a), and its
factor may carry one rounding of 1 / |e|, no more."""
import numpy as np
import pytest

from imodel_amd.swm import ERAD_REF, GRAV, Mesh, Swm

pytestmark = pytest.mark.gpu

SCHEMES = {"plain": {}, "hc": {"stag": "HC"}, "apvm": {"pv": "apvm", "pvspar": 0.5}, "pxt16": {"wrap": "pxt16"},
           "k2": {"k2": 1e5, "diffus": "const"}}


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("scheme", list(SCHEMES))
def test_gradient_factor(scheme, prec):
    """Cells one metre deeper than the rest, no two of them neighbours: the
    jump of the potential is that of one metre at each of their edges, a number
    of the handle's type, so momeq is its product with 1 / |e| rounded to that
    type, bit for bit."""
    print("[gpu-case] stage gradient", scheme, prec, flush=True)
    m = Mesh.icos(4)
    a = m.arrays
    ends = a["ed_v"].reshape(-1, 2) - 1
    near = [[] for _ in range(m.nv)]
    for i, j in ends:
        near[i].append(j)
        near[j].append(i)
    deep = np.zeros(m.nv, dtype=bool)
    for i in range(m.nv):
        deep[i] = not any(deep[j] for j in near[i])
    h = np.where(deep, 1001.0, 1000.0)
    with Swm(m, precision=prec, h_ref=1000.0) as s:
        s.set_scheme(**SCHEMES[scheme])
        _, f = s.tendency(h, np.zeros(m.ne))
        assert list(s.profile(1)) == ["fast_stage"]
    T = np.float32 if prec == "fp32" else np.float64
    jump = T(GRAV) * T(1.0 / ERAD_REF)
    edge = deep[ends[:, 0]] != deep[ends[:, 1]]
    assert edge.sum() > 2000 and not np.any(f[~edge])
    want = jump * (1.0 / a["ed_leng"][edge]).astype(T)
    assert want.dtype == T and np.array_equal(np.abs(f[edge]), want.astype(np.float64))
